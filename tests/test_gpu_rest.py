"""Bottom-up levels with few vertices left: chunks with none, one and many entries, more entries
than a round of lanes takes, vertices found and missed side by side."""
import numpy as np
import pytest
from scipy.sparse import coo_matrix
from scipy.sparse.csgraph import dijkstra

import g500bfs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counting", [False, True])
@pytest.mark.parametrize("pairs,tails", [(0, 0), (0, 300), (40, 40), (700, 0), (400, 400)])
def test_levels(pairs, tails, counting):
    small = G.Graph.generate(17, 8)
    v0, v1 = small.edges()
    small.free()
    n = 1 << 17
    used = np.unique(np.concatenate([v0, v1]))
    # the vertices of one degree are neighbours in the engine's order: components of one edge and
    # tails of three vertices, interleaved, above all other IDs
    ids = n + np.arange(2 * pairs + 3 * tails)
    a, b = [v0], [v1]
    pair = ids[:2 * pairs].reshape(-1, 2)
    a.append(pair[:, 0]), b.append(pair[:, 1])
    tail = ids[2 * pairs:].reshape(-1, 3)
    at = used[np.linspace(0, len(used) - 1, tails).astype(np.int64)] if tails else used[:0]
    for x, y in ((at, tail[:, 0]), (tail[:, 0], tail[:, 1]), (tail[:, 1], tail[:, 2])):
        a.append(x), b.append(y)
    a, b = np.concatenate(a), np.concatenate(b)
    total = n + len(ids)
    adj = coo_matrix((np.ones(len(a), np.int8), (a, b)), shape=(total, total)).tocsr()
    g = G.Graph.from_edges(a, b).construct()
    bfs = G.Bfs(g)
    bfs.set_counting(counting)
    for root in g.find_roots(2):
        depth = dijkstra(adj, directed=False, indices=int(root), unweighted=True)
        want = np.where(np.isinf(depth), 0xFFFF, depth).astype(np.uint16)
        for beta in (14.0, 1e7):  # 1e7: bottom-up to the end
            bfs.run(int(root), edgefactor=8, beta=beta)
            np.testing.assert_array_equal(bfs.levels()[:total], want)
            assert bfs.validate(int(root))[0]
    bfs.destroy()
    g.free()
