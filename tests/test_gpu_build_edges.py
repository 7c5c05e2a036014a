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


def _same_csr(G, v0, v1, **flags):
    og = O.Graph(np.asarray(v0, np.int64), np.asarray(v1, np.int64))
    if flags.get("symmetric_input"):
        v0, v1 = np.concatenate([v0, v1]), np.concatenate([v1, v0])
    g = G.Graph.from_edges(v0, v1).construct(**flags)
    i, o = g.info, og.info
    assert (i.log_n, i.n, i.n_c, i.m, i.m_sym, i.max_used_vertex) == (
        o.log_n, o.n, o.n_c, o.m, o.m_sym, o.max_used_vertex)
    a, b = g.csr(), og.arrays()
    for k in ("row_off", "col", "deg_new", "new2orig", "orig2new"):
        assert np.array_equal(a[k].astype(np.int64), b[k].astype(np.int64)), k
    return g


def _skewed(vertices, edges, seed):
    rng = np.random.default_rng(seed)
    v = np.zeros((2, edges), np.int64)
    for _ in range(max(1, (vertices - 1).bit_length())):
        r = rng.random(edges)
        src = r >= 0.76
        v[0] = 2 * v[0] + src
        v[1] = 2 * v[1] + (((r >= 0.57) & ~src) | (r >= 0.95))
    return rng.permutation(vertices)[v % vertices]


# keys are laid out 3072 a bucket (1536 edges) and sorted up to 4096 a time,
# one partition pass up to 2048 buckets (3145728 edges), two beyond; tiles of
# 8192 keys
@pytest.mark.parametrize("vertices,edges", [
    (2, 1), (5, 3), (100, 1535), (100, 1536), (100, 1537), (100, 2047), (100, 2048), (100, 2049),
    (3000, 4096), (3000, 4097), (200003, 3145727), (200003, 3145731),
    (70001, 300007),          # two ID ranges of 2^16
    (1048577, 1100001),       # IDs past 2^20: endpoints partitioned before they are counted
    (300007, 4194305),        # one key pair more than one pass holds
    (600011, 6000001)])
@pytest.mark.parametrize("symmetric", [False, True])
def test_rows_of_skewed_lists(G, vertices, edges, symmetric):
    print(f"\n[build] {vertices} vertices {edges} edges symmetric={symmetric}", flush=True)
    v0, v1 = _skewed(vertices, edges, edges)
    _same_csr(G, v0, v1, symmetric_input=symmetric)


@pytest.mark.parametrize("shape", [
    "star",        # one row of 70000 targets of degree 1: its counter passes 2^15 twice
    "repeated",    # every key the same: no bucket bound can part them
    "loops",       # nothing but loops
    "hubs",        # rows of 3000 to 9000 entries among short ones
    "bipartite",   # two hubs whose targets all lie at one end of the order
    "sparse",      # few edges over IDs up to 2^27
    "wide"])       # hub rows over IDs up to 2^27: 54 key bits, no room for the bucket number in a key
def test_rows_of_odd_lists(G, shape):
    print(f"\n[build] {shape}", flush=True)
    rng = np.random.default_rng(11)
    if shape == "star":
        v0, v1 = np.full(70000, 70000, np.int64), np.arange(70000, dtype=np.int64)
    elif shape == "repeated":
        v0, v1 = np.full(40000, 3, np.int64), np.full(40000, 9, np.int64)
    elif shape == "loops":
        v0 = np.concatenate([np.full(50000, 6, np.int64), [1]])
        v1 = np.concatenate([np.full(50000, 6, np.int64), [2]])
    elif shape == "hubs":
        v0 = np.concatenate([np.full(3000 + 1000 * i, i, np.int64) for i in range(7)]
                            + [rng.integers(0, 50000, 100000)])
        v1 = rng.integers(0, 50000, len(v0))
    elif shape == "bipartite":
        a = np.arange(30000, dtype=np.int64) + 10
        v0 = np.concatenate([np.full(30000, 0, np.int64), np.full(30000, 1, np.int64)])
        v1 = np.concatenate([a, a])
    elif shape == "sparse":
        v0, v1 = rng.integers(0, 1 << 27, 5000), rng.integers(0, 1 << 27, 5000)
    else:
        v0, v1 = rng.integers(0, 1 << 27, 40000), rng.integers(0, 40, 40000)
    _same_csr(G, v0, v1)
