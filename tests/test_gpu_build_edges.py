"""GPU construction at the edges of its tiles, against the oracle, bit for bit."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import g500bfs
    g500bfs.load()
    return g500bfs


def _ring(n, first=0):
    i = np.arange(n, dtype=np.int64)
    return first + i, first + (i + 1) % n


# a ring of L vertices has 2 L CSR entries; the core filter takes them 2048 a tile
@pytest.mark.parametrize("ring,pendants,spokes", [
    (3, 0, 0), (1023, 1, 0), (1024, 0, 0), (1024, 1, 0), (1025, 7, 0), (2047, 3, 0),
    (700, 900, 0),      # as many pendants as ring vertices: most entries go
    (5000, 11, 5000),   # a hub row over several tiles, all of it kept
    (5000, 6000, 3)])   # a hub row over several tiles, nearly all of it pruned
def test_core_filter_tiles(G, ring, pendants, spokes):
    print(f"\n[build] core filter ring={ring} pendants={pendants} spokes={spokes}", flush=True)
    v0, v1 = _ring(ring)
    hub = ring
    p = np.arange(pendants, dtype=np.int64) + ring + 1
    on = np.full(pendants, hub) if spokes else np.arange(pendants) % ring
    s = np.arange(spokes, dtype=np.int64)
    v0 = np.concatenate([v0, on, np.full(spokes, hub, np.int64)]).astype(np.int64)
    v1 = np.concatenate([v1, p, s]).astype(np.int64)
    cb = O.Graph(v0, v1).corebfs()
    g = G.Graph.from_edges(v0, v1).construct(corebfs=True)
    bfs = G.Bfs(g)
    inf = g.refresh().info
    assert (inf.core_vertices, inf.m) == (cb["core_vertices"], cb["core_edges"])
    assert inf.tree_vertices == cb["tree_vertices"] and inf.removed_parents == cb["removed"]
    tp, hp = g.forest()
    assert np.array_equal(tp, cb["tree_parent"]) and np.array_equal(hp, cb["has_parent"])
    at = bfs.run(0)
    ok, _, errs = bfs.validate(0)
    assert ok, (errs, at)
