"""Runs in one block against the oracle and against the level loop."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import g500bfs
    g500bfs.load()
    return g500bfs


def _run(bfs, root, **kw):
    at = bfs.run(root, **kw)
    _, trace = bfs.stats()
    lev = bfs.levels()
    ok, te, errs = bfs.validate(root)
    assert ok, errs
    return at.tolist(), [(t["level"], t["top_down"], t["nq_size"], t["nq_edges"],
                          t["exec_bottom_up"]) for t in trace], lev, te


# an engine that times its levels takes the level loop: same directions,
# frontiers and levels from both; SCALE 15 is past the one block's vertices
@pytest.mark.parametrize("scale,edgefactor", [(5, 16), (8, 3), (10, 16), (12, 16), (13, 31),
                                              (14, 16), (14, 5), (15, 16)])
@pytest.mark.parametrize("exec_alpha", [25.0, 0.0, 1e9])
def test_same_run_as_the_level_loop(G, scale, edgefactor, exec_alpha):
    print(f"\n[small] scale {scale} ef {edgefactor} exec_alpha {exec_alpha}", flush=True)
    g = G.Graph.generate(scale, edgefactor).construct()
    one, loop = G.Bfs(g), G.Bfs(g)
    loop.set_timing(True)
    for b in (one, loop):
        b.set_exec_alpha(exec_alpha)
    for r in g.find_roots(4).tolist():
        for alpha, beta in ((10.0, 14.0), (1e9, 14.0), (1e-9, 14.0), (4.0, 1e9)):
            kw = dict(edgefactor=edgefactor, alpha=alpha, beta=beta)
            a, b = _run(one, r, **kw), _run(loop, r, **kw)
            assert a[:2] == b[:2] and np.array_equal(a[2], b[2]) and a[3] == b[3]


def _chain(n):
    v = np.arange(n, dtype=np.int64)
    return v[:-1], v[1:]


# chains around the most steps one block takes (the level loop runs beyond),
# stars, a clique with a long row, vertex counts at the edges of words
@pytest.mark.parametrize("name,v0,v1", [
    ("edge", *_chain(2)), ("chain 33", *_chain(33)), ("chain 60", *_chain(60)),
    ("chain 63", *_chain(63)), ("chain 64", *_chain(64)), ("chain 300", *_chain(300)),
    ("star", np.zeros(5000, np.int64), np.arange(1, 5001)),
    ("far star", np.concatenate([np.zeros(16000, np.int64), [1, 16001]]),
     np.concatenate([np.arange(1, 16001), [16001, 16002]])),
    ("clique", *(x.ravel() for x in np.meshgrid(np.arange(200), np.arange(200)))),
    ("16384", *_chain(40)), ])
def test_odd_graphs(G, name, v0, v1):
    print(f"\n[small] {name}", flush=True)
    if name == "16384":  # as many vertices as one block holds, half of them far
        v0 = np.concatenate([v0, np.arange(40, 16384) % 40, np.arange(100, 8292)])
        v1 = np.concatenate([v1, np.arange(40, 16384), np.arange(8292, 16484) - 100])
    v0, v1 = np.asarray(v0, np.int64), np.asarray(v1, np.int64)
    g = G.Graph.from_edges(v0, v1).construct()
    og = O.Graph(v0, v1)
    bfs = G.Bfs(g)
    for root in (int(v0[0]), int(v1[-1])):
        for alpha in (10.0, 1e9):
            ref = og.bfs(root)
            _, _, lev, _ = _run(bfs, root, alpha=alpha)
            assert np.array_equal(lev, np.where(ref < 0, 0xFFFF, ref).astype(np.uint16))


def test_after_a_root_without_edges(G):
    print("\n[small] isolated root", flush=True)
    g = G.Graph.from_edges(np.array([0, 1, 6]), np.array([1, 2, 7])).construct()
    bfs = G.Bfs(g)
    for root, want in ((4, [4]), (0, [0, 1, 2]), (5, [5]), (6, [6, 7]), (2, [2, 1, 0])):
        bfs.run(root)
        assert sorted(np.nonzero(bfs.levels() != 0xFFFF)[0].tolist()) == sorted(want)
        assert bfs.pred()[root] == root
