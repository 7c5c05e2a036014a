"""When the validator orders a graph's edges: the second pass over them, not the first."""
import threading

import numpy as np
import pytest

import oracle_lib as O
from test_gpu_validate_tiles import _entry

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import g500bfs
    g500bfs.load()
    return g500bfs


# 2^20 edges at least: large enough for the order
@pytest.mark.parametrize("scale,corebfs", [(16, False), (18, False), (18, True)])
def test_ordered_by_the_second_pass(G, golden, scale, corebfs):
    print(f"\n[order] scale {scale} corebfs={corebfs}", flush=True)
    g = G.Graph.generate(scale).construct(corebfs=corebfs)
    a, b = G.Bfs(g), G.Bfs(g)
    root = int(g.find_roots(1)[0])
    held, copy = g.refresh().info.device_bytes, 8 * g.info.nedges_input

    def check(bfs):
        bfs.run(root)
        ok, te, errs = bfs.validate(root)
        assert ok and te == golden["pf_nedge"][scale], errs
        return g.refresh().info.device_bytes - held

    assert check(a) == 0  # one tree of a graph: the direct pass
    # a tree that fails before its edges are looked at does not count
    pred = a.pred()
    pred[root] = -1
    for _ in range(3):
        ok, _, errs = a.validate(root, host_pred=pred)
        assert not ok
    assert g.refresh().info.device_bytes == held
    assert check(b) >= copy  # another engine's second pass: the copy, kept with the graph
    assert check(a) == check(b)


# trees deeper than the codes hold take the direct pass every time
def test_deep_trees_are_never_ordered(G):
    print("\n[order] deep", flush=True)
    v0 = np.tile(np.arange(40, dtype=np.int64), 30000)
    g = G.Graph.from_edges(v0, v0 + 1).construct()
    bfs = G.Bfs(g)
    held = g.info.device_bytes
    for _ in range(3):
        bfs.run(0)
        ok, te, errs = bfs.validate(0)
        assert ok and te == len(v0), errs
    assert g.refresh().info.device_bytes == held


# mistakes in a tree that the direct pass, the ordering one and a later one check
def test_mistakes_before_and_after(G):
    print("\n[order] mistakes", flush=True)
    scale = 17
    g = G.Graph.generate(scale).construct()
    og = O.Graph(*O.generate_edges(scale))
    bfs = G.Bfs(g)
    r = int(g.find_roots(1)[0])
    bfs.run(r)
    pred, lev = bfs.pred(), og.bfs(r)
    parents = set(((pred[lev > 0] << 16) >> 16).tolist())
    leaves = [int(v) for v in np.nonzero(lev > 1)[0] if int(v) not in parents]
    bad = pred.copy()
    bad[leaves[0]] = -1
    deep = int(lev.max())
    w = next(x for x in leaves if lev[x] == deep - 1)
    bad[w] = _entry(next(int(x) for x in np.nonzero(lev == deep - 1)[0] if int(x) != w), deep)
    ok_o, te_o, errs_o = og.validate(r, bad)
    for _ in range(4):
        ok, te, errs = bfs.validate(r, host_pred=bad)
        assert not ok and not ok_o
        assert te == te_o and list(errs.values()) == [int(errs_o[k]) for k in errs], errs
        ok, te, errs = bfs.validate(r, host_pred=pred)
        assert ok and te == og.validate(r, pred)[1], errs


# engines of one graph: one of them orders while the others pass directly
def test_engines_side_by_side(G, golden):
    print("\n[order] threads", flush=True)
    scale = 20
    g = G.Graph.generate(scale).construct()
    engines = [G.Bfs(g) for _ in range(3)]
    roots = g.find_roots(3).tolist()
    wrong = []

    def work(bfs, root):
        for _ in range(4):
            bfs.run(root)
            ok, te, errs = bfs.validate(root)
            if not ok or te != golden["pf_nedge"][scale]:
                wrong.append((root, te, errs))

    ts = [threading.Thread(target=work, args=x) for x in zip(engines, roots)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong
