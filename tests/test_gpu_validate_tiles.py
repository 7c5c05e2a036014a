"""The validator's ordered-edge pass against the oracle and plain counts."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import g500bfs
    g500bfs.load()
    return g500bfs


def _entry(parent, depth):
    u = (int(depth) << 48) | (int(parent) & 0xFFFFFFFFFFFF)
    return np.int64(u - (1 << 64) if u >= 1 << 63 else u)


# SCALE 16: one tile of edges, SCALE 18: two slices of sources
@pytest.mark.parametrize("scale", [16, 18])
def test_planted_mistakes_counted_alike(G, scale):
    print(f"\n[validate] planted, scale {scale}", flush=True)
    g = G.Graph.generate(scale).construct()
    og = O.Graph(*O.generate_edges(scale))
    bfs = G.Bfs(g)
    r = int(g.find_roots(1)[0])
    bfs.run(r)
    pred, lev = bfs.pred(), og.bfs(r)
    parents = set(((pred[lev > 0] << 16) >> 16).tolist())
    leaves = [int(v) for v in np.nonzero(lev > 1)[0] if int(v) not in parents]
    plants = {}
    p = pred.copy()
    p[leaves[0]] = -1  # unreached beside reached neighbours
    plants["tree"] = p
    p = pred.copy()  # a parent at the right depth that is no neighbour
    v = leaves[1]
    e0, e1 = g.edges()
    near = set(e1[e0 == v].tolist()) | set(e0[e1 == v].tolist())
    p[v] = _entry(next(int(w) for w in np.nonzero(lev == lev[v] - 1)[0] if int(w) not in near),
                  lev[v])
    plants["no edge"] = p
    p = pred.copy()  # a whole branch one level too deep, right among itself
    deep = int(lev.max())
    w = next(int(x) for x in leaves if lev[x] == deep - 1)
    p[w] = _entry(next(int(x) for x in np.nonzero(lev == deep - 1)[0] if int(x) != w), deep)
    plants["gap or no edge"] = p
    for name, p in plants.items():
        ok, te, errs = bfs.validate(r, host_pred=p)
        ok_o, te_o, errs_o = og.validate(r, p)
        assert not ok and not ok_o, name
        assert te == te_o and list(errs.values()) == [int(errs_o[k]) for k in errs], (name, errs, errs_o)
    ok, te, errs = bfs.validate(r, host_pred=pred)
    assert ok and te == og.validate(r, pred)[1], errs


# IDs up to 2^25 make 4096 tiles, ordered in two passes; loops name IDs past
# the last vertex with an edge
def test_two_pass_order(G):
    print("\n[validate] two passes", flush=True)
    rng = np.random.default_rng(3)
    v0, v1 = rng.integers(0, 1 << 25, (2, 1500001))
    v0[:600000], v1[:600000] = rng.integers(0, 4000, (2, 600000))
    v1[600000:700000] = v0[600000:700000]
    g = G.Graph.from_edges(v0, v1).construct()
    bfs = G.Bfs(g)
    root = int(v0[np.argmax(v0 != v1)])
    bfs.run(root)
    lev = bfs.levels()
    for _ in range(2):
        ok, te, errs = bfs.validate(root)
        assert ok, errs
        assert te == int((lev[v0] != 0xFFFF).sum())


# deeper than the codes hold: the direct pass
def test_deep_tree(G):
    print("\n[validate] deep", flush=True)
    v0 = np.tile(np.arange(40, dtype=np.int64), 30000)
    g = G.Graph.from_edges(v0, v0 + 1).construct()
    bfs = G.Bfs(g)
    bfs.run(0)
    ok, te, errs = bfs.validate(0)
    assert ok and te == len(v0), errs


def test_corebfs_depths_rebuilt(G, golden):
    print("\n[validate] CoreBFS", flush=True)
    g = G.Graph.generate(18).construct(corebfs=True)
    bfs = G.Bfs(g)
    for r in g.find_roots(4).tolist():
        bfs.run(r)
        ok, te, errs = bfs.validate(r)
        assert ok and te == golden["pf_nedge"][18], errs
