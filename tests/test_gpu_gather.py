"""pred by original ID: words with every, no and some vertices with edges, a last word that is not
full, roots inside and outside the lists."""
import numpy as np
import pytest

import g500bfs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 64, 65, 511, 513, 8 * 64 * 8 + 1, 40961])
@pytest.mark.parametrize("step", [1, 2, 67])
def test_pred_of_a_path(n, step):
    """A path over every `step`-th of the first n IDs; the others have no edges."""
    ids = np.arange(0, n, step, dtype=np.int64)[:60]
    far = np.arange(n - 1, n - 1 - min(n // 2, 200), -1, dtype=np.int64)  # leaves of ids[0]
    far = far[far > ids[-1]]
    v0 = np.concatenate([ids[:-1], np.full(len(far), ids[0], dtype=np.int64)])
    v1 = np.concatenate([ids[1:], far])
    g = G.Graph.from_edges(v0, v1).construct()
    b = G.Bfs(g)
    b.set_timing(True)  # the level loop
    depth = np.full(len(g_pred(b, int(ids[0]))), -1, dtype=np.int64)
    depth[ids] = np.arange(len(ids))
    depth[far] = 1
    lone = [v for v in range(min(n, 130)) if depth[v] < 0][:1]
    for root in [int(ids[0])] + lone + [int(ids[0])]:
        pred = g_pred(b, root)
        if root in lone:
            assert pred[root] == root
            assert (np.delete(pred, root) == -1).all()
            continue
        reached = depth >= 0
        assert (pred[~reached] == -1).all()
        parent, level = pred[reached] & ((1 << 48) - 1), pred[reached] >> 48
        np.testing.assert_array_equal(level, depth[reached])
        below = level > 0
        np.testing.assert_array_equal(depth[parent[below]], level[below] - 1)
        assert parent[~below] == root
    b.destroy()
    g.free()


def g_pred(b, root):
    b.run(root)
    return b.pred()


@pytest.mark.parametrize("guess", ["", "wrong"])
@pytest.mark.parametrize("corebfs", [False, True])
@pytest.mark.parametrize("stride", [1, 64, 128, 129])  # vertices: 2^16, 2^22, 2^23, over 2^23
def test_gather_beside_and_behind_the_levels(stride, corebfs, guess, monkeypatch):
    """The same tree whether the gather runs beside the last levels (large graphs) or ends the
    run."""
    if guess:
        monkeypatch.setenv("G500_GUESS", guess)
    small = G.Graph.generate(16)
    v0, v1 = small.edges()
    g = G.Graph.from_edges(v0 * stride, v1 * stride).construct(corebfs=corebfs)
    small.construct(corebfs=corebfs)
    b, ref = G.Bfs(g), G.Bfs(small)
    for root in small.find_roots(4):
        ref.run(int(root))
        for _ in range(2):
            b.run(int(root) * stride)
            levels = b.levels()
            np.testing.assert_array_equal(levels[:stride << 16:stride], ref.levels())
            assert (np.delete(levels, np.s_[:stride << 16:stride]) == 0xFFFF).all()
            assert b.validate(int(root) * stride)[0]
    for x in (b, ref):
        x.destroy()
    for x in (g, small):
        x.free()
