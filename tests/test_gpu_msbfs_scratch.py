"""What creating a batched engine takes of the device, and its input-edge counts."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import g500bfs
    g500bfs.load()
    return g500bfs


def _free_bytes():
    hip = C.CDLL("libamdhip64.so.7")  # the one the library runs on
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _te(v0, levels, n):
    """Input edges whose source the root reaches (sources from n on are loops outside)."""
    return int((levels[v0[v0 < n]] != 0xFFFF).sum())


# loops may name any ID: the graph keeps the vertices of the other edges only.
# What creation takes, kept scratch included, stays near the footprint
@pytest.mark.parametrize("vertices,edges,far", [
    (1000, 5000, 1 << 30), (1000, 5000, (1 << 30) + 12345), (60000, 400000, 1 << 29),
    (70000, 200000, 131072), (300, 100, 511), (2000000, 3000000, 1 << 30)])
def test_loops_at_far_ids(G, vertices, edges, far):
    print(f"\n[msbfs] {vertices} vertices {edges} edges, loops from {far}", flush=True)
    rng = np.random.default_rng(edges)
    v0, v1 = rng.integers(0, vertices, (2, edges))
    loops = far + rng.integers(0, 64, 1000)
    near = rng.integers(0, vertices, 500)
    v0, v1 = np.concatenate([v0, loops, near]), np.concatenate([v1, loops, near])
    order = rng.permutation(len(v0))
    v0, v1 = v0[order], v1[order]
    g = G.Graph.from_edges(v0, v1).construct()
    bfs = G.Bfs(g)
    roots = g.find_roots(4)
    G.device_memory()
    before = _free_bytes()
    batch = G.MultiBfs(g, max_roots=4)
    taken = before - _free_bytes()
    assert taken <= G.msbfs_footprint(g, 4) + (128 << 20), taken
    batch.run(roots)
    te = batch.te()
    for i, r in enumerate(roots.tolist()):
        bfs.run(r)
        levels = bfs.levels()
        assert np.array_equal(batch.levels(i), np.where(levels == 0xFFFF, 0xFF, levels).astype(np.uint8))
        assert te[i] == _te(v0, levels, g.info.n)


# sources counted in one range of IDs, in several directly, and partitioned
@pytest.mark.parametrize("scale,edgefactor", [(10, 16), (17, 16), (21, 4), (21, 16), (18, 1)])
def test_counts_of_every_form(G, scale, edgefactor):
    print(f"\n[msbfs] counts, scale {scale} edge factor {edgefactor}", flush=True)
    g = G.Graph.generate(scale, edgefactor).construct()
    v0, _ = g.edges()
    bfs, batch = G.Bfs(g), G.MultiBfs(g, max_roots=3)
    roots = g.find_roots(3)
    batch.run(roots)
    te = batch.te()
    for i, r in enumerate(roots.tolist()):
        bfs.run(r)
        assert te[i] == _te(v0, bfs.levels(), g.info.n)


def test_footprint_covers_the_counting(G):
    print("\n[msbfs] footprint", flush=True)
    for scale, ef in ((20, 4), (20, 64), (22, 32)):
        g = G.Graph.generate(scale, ef).construct()
        need = G.msbfs_footprint(g, 1, level_arrays=False)
        assert need >= 8 * g.info.n + 2 * g.info.nedges_input
