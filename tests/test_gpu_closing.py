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
