"""The last block of a step's last kernel closes it: blocks that take part from one, over one
ticket slot each, to the whole grid."""
import numpy as np
import pytest

import g500bfs as G

pytestmark = pytest.mark.gpu

TILE, SLOTS, GRID = 2048, 64, 2048  # edges per tile, ticket slots, blocks


@pytest.mark.parametrize("leaves", [1, TILE, TILE + 1, SLOTS * TILE, SLOTS * TILE + 1,
                                    (SLOTS + 1) * TILE + 1, GRID * TILE, GRID * TILE + 1])
def test_star(leaves):
    hub = 5
    v1 = np.arange(leaves + 1, dtype=np.int64)
    v1 = v1[v1 != hub] if leaves >= hub else np.arange(hub + 1, hub + 1 + leaves)
    g = G.Graph.from_edges(np.full(len(v1), hub, dtype=np.int64), v1).construct()
    b = G.Bfs(g)
    b.set_timing(True)  # the level loop, also where one block could run it all
    for root in (hub, int(v1[-1])):
        for _ in range(2):
            b.run(root)
            levels = b.levels()
            want = np.full(len(levels), 0xFFFF, dtype=levels.dtype)
            want[v1] = 1 if root == hub else 2
            want[hub] = 0 if root == hub else 1
            want[root] = 0
            np.testing.assert_array_equal(levels, want)
    b.destroy()
    g.free()


@pytest.mark.parametrize("tiles", [7, 8, 9, 10, 70])
@pytest.mark.parametrize("extra", [-1, 0, 1])
@pytest.mark.parametrize("hubs", [1, 3])
def test_frontier_with_hubs(tiles, extra, hubs):
    """A frontier of 600 vertices (prepared by the prefix-sum launches) of which some own about
    `tiles` tiles of edges and the others one edge."""
    mid, leaves = 600, tiles * TILE + extra
    v0, v1 = [np.zeros(mid, np.int64)], [np.arange(1, mid + 1)]
    nxt = mid + 1
    for h in range(hubs):
        v0.append(np.full(leaves, 1 + h * (mid - 1) // max(hubs - 1, 1), np.int64))
        v1.append(np.arange(nxt, nxt + leaves))
        nxt += leaves
    v0.append(np.arange(1, mid + 1)), v1.append(np.arange(nxt, nxt + mid))
    nxt += mid
    g = G.Graph.from_edges(np.concatenate(v0), np.concatenate(v1)).construct()
    b = G.Bfs(g)
    b.set_exec_alpha(0)  # the heavy level is expanded, not swept
    b.set_timing(True)
    for _ in range(2):
        b.run(0, alpha=1e-3)  # top-down to the end
        levels = b.levels()
        want = np.full(len(levels), 0xFFFF, dtype=levels.dtype)
        want[0], want[1:mid + 1], want[mid + 1:nxt] = 0, 1, 2
        np.testing.assert_array_equal(levels, want)
        assert b.validate(0)[0]
    b.destroy()
    g.free()
