"""The level loop on graphs that otherwise run in one block: partial words, chunks and tiles."""
import numpy as np
import pytest

import oracle_lib as O
from test_gpu_parity import _small_cases

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import g500bfs
    g500bfs.load()
    return g500bfs


# runs that time their levels, and runs that count their bytes, take the loop
LOOP = {"timing": lambda bfs: bfs.set_timing(True), "counting": lambda bfs: bfs.set_counting(True)}


def _u16(ref):
    return np.where(ref < 0, 0xFFFF, ref).astype(np.uint16)


def _check(G, g, og, roots, how, settings):
    block, loop = G.Bfs(g), G.Bfs(g)
    LOOP[how](loop)
    sweeps = 0
    for root in roots:
        ref = _u16(og.bfs(int(root)))
        for alpha, beta, exec_alpha in settings:
            for b in (block, loop):
                b.set_exec_alpha(exec_alpha)
            want = block.run(int(root), 16, alpha, beta)
            at = loop.run(int(root), 16, alpha, beta)
            assert np.array_equal(at, want), (root, alpha, beta)
            assert np.array_equal(loop.levels(), ref), (root, alpha, beta)
            ok, _, errs = loop.validate(int(root))
            assert ok, errs
            pred = loop.pred()
            found = ref != 0xFFFF
            assert np.array_equal(pred == -1, ~found)
            stats, trace = loop.stats()
            sweeps += stats.sweeps
            assert [(t["level"], t["nq_size"], t["nq_edges"], t["top_down"]) for t in trace] == \
                [(t["level"], t["nq_size"], t["nq_edges"], t["top_down"]) for t in block.stats()[1]]
    return sweeps


# (alpha, beta, exec_alpha): the defaults, bottom-up from the second level on,
# the same to the end, top-down throughout by expansion, and there as sweeps
SETTINGS = [(10.0, 14.0, 25.0), (1e9, 14.0, 25.0), (1e9, 1e6, 25.0), (1e-3, 14.0, 0.0),
            (1e-3, 14.0, 1e9)]


@pytest.mark.parametrize("how", list(LOOP))
@pytest.mark.parametrize("vertices", [3, 63, 64, 65, 511, 512, 513, 1025, 4095, 4097, 16384])
def test_chunk_edges(G, vertices, how):
    print(f"\n[loop] {vertices} vertices {how}", flush=True)
    rng = np.random.default_rng(vertices)
    # every vertex hangs on a random earlier one and on a few others
    v0 = np.arange(1, vertices, dtype=np.int64)
    v1 = (rng.random(vertices - 1) * v0).astype(np.int64)
    extra = rng.integers(0, vertices, (2, 3 * vertices))
    v0, v1 = np.concatenate([v0, extra[0]]), np.concatenate([v1, extra[1]])
    g = G.Graph.from_edges(v0, v1).construct()
    sweeps = _check(G, g, O.Graph(v0, v1), (0, int(v0[-1])), how, SETTINGS)
    assert sweeps > 0


@pytest.mark.parametrize("how", list(LOOP))
@pytest.mark.parametrize("name", list(_small_cases()))
def test_small_cases(G, name, how):
    print(f"\n[loop] {name} {how}", flush=True)
    v0, v1 = (np.asarray(x, np.int64) for x in _small_cases()[name])
    g = G.Graph.from_edges(v0, v1).construct()
    og = O.Graph(v0, v1)
    roots = [v for v in range(og.info.n) if og.has_edge(v)][:5]
    _check(G, g, og, roots, how, SETTINGS)


@pytest.mark.parametrize("how", list(LOOP))
@pytest.mark.parametrize("alpha,beta", [(1e9, 14.0), (1e-3, 14.0), (10.0, 1e-6), (0.5, 1e6)])
def test_direction_extremes(G, alpha, beta, how):
    print(f"\n[loop] alpha={alpha} beta={beta} {how}", flush=True)
    g = G.Graph.generate(14).construct()
    og = O.Graph(*O.generate_edges(14))
    _check(G, g, og, g.find_roots(3).tolist(), how, [(alpha, beta, 25.0)])


def test_top_down_throughout(G):
    """Large frontiers expanded top-down at every level: block prefix sums, a last-block scan of
    their totals, tile owners."""
    print("\n[loop] scale 18 top-down", flush=True)
    g = G.Graph.generate(18).construct()
    og = O.Graph(*O.generate_edges(18))
    bfs = G.Bfs(g)
    bfs.set_exec_alpha(0)
    for root in g.find_roots(3).tolist():
        bfs.run(root, 16, 1e-3, 14.0)
        assert np.array_equal(bfs.levels(), _u16(og.bfs(root)))
        ok, _, errs = bfs.validate(root)
        assert ok, errs
        trace = bfs.stats()[1]
        assert all(t["top_down"] and not t["exec_bottom_up"] for t in trace)
        sizes = [t["nq_size"] for t in trace]
        assert max(sizes) > 65536 and any(512 < s <= 65536 for s in sizes)
