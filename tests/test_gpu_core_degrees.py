"""Degrees counted from the rows of a CSR: a graph without trees is its own core, whose rows must
come out as the plain construction's do."""
import numpy as np
import pytest

import g500bfs as G

pytestmark = pytest.mark.gpu


def cycle(n, first):
    v = first + np.arange(n)
    return v, np.roll(v, -1)


def clique(n, first):
    a, b = np.triu_indices(n, 1)
    return first + a, first + b


@pytest.mark.parametrize("parts", [
    [(cycle, 3)], [(cycle, 127)], [(cycle, 128)], [(cycle, 129)], [(cycle, 1024)],
    [(cycle, 1025)], [(clique, 3)], [(clique, 65)], [(clique, 700)], [(clique, 2200)],
    [(cycle, 100003), (clique, 300), (cycle, 5)], [(clique, 64)] * 100,
])
def test_core_of_a_graph_without_trees(parts):
    v0, v1, first = [], [], 1
    for kind, n in parts:
        a, b = kind(n, first)
        v0.append(a), v1.append(b)
        first += n + 3
    v0, v1 = np.concatenate(v0), np.concatenate(v1)
    # some edges twice and, as loops, some vertices
    v0, v1 = np.concatenate([v0, v1[::3], v0[::5]]), np.concatenate([v1, v0[::3], v0[::5]])
    plain = G.Graph.from_edges(v0, v1).construct()
    core = G.Graph.from_edges(v0, v1).construct(corebfs=True)
    assert core.info.n_c == plain.info.n_c and core.info.m == plain.info.m
    edges = []
    for x in (plain.csr(), core.csr()):
        size = np.diff(x["row_off"])
        src = x["new2orig"][np.repeat(np.arange(len(size)), size)].astype(np.int64)
        edges.append(np.sort(src << 32 | x["new2orig"][x["col"]]))
    np.testing.assert_array_equal(*edges)
    # without repeated edges a degree is the row's length
    np.testing.assert_array_equal(x["deg_new"], size)
    root = int(v0[0])
    b, c = G.Bfs(plain), G.Bfs(core)
    b.run(root), c.run(root)
    np.testing.assert_array_equal(b.levels(), c.levels())
    assert c.validate(root)[0]
    for x in (b, c):
        x.destroy()
    for x in (plain, core):
        x.free()
