"""Lists that cannot be bucketed take the general sort, against the oracle, bit for bit."""
import numpy as np
import pytest

from test_gpu_build_edges import _same_csr, _skewed

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import g500bfs
    g500bfs.load()
    return g500bfs


# a bucket may hold 65536 keys: one key just as often, once more, and many times
# more (one direction a bucket where the list holds both)
@pytest.mark.parametrize("times", [65535, 65536, 65537, 300000])
@pytest.mark.parametrize("rest", [0, 20000])
@pytest.mark.parametrize("symmetric", [False, True])
def test_one_edge_repeated(G, times, rest, symmetric):
    print(f"\n[general] {times} times, {rest} others, symmetric={symmetric}", flush=True)
    rng = np.random.default_rng(times + rest)
    v0 = np.concatenate([np.full(times, 17), rng.integers(0, 3000, rest)]).astype(np.int64)
    v1 = np.concatenate([np.full(times, 5), rng.integers(0, 3000, rest)]).astype(np.int64)
    order = rng.permutation(len(v0))
    _same_csr(G, v0[order], v1[order], symmetric_input=symmetric)


# over 3145728 edges the keys go through groups first: repeated pairs past one
# group's room, and a hub whose targets all lie in one
@pytest.mark.parametrize("shape", ["pair", "pairs", "hub"])
def test_groups_past_their_room(G, shape):
    print(f"\n[general] groups, {shape}", flush=True)
    rng = np.random.default_rng(7)
    v0, v1 = _skewed(100003, 3000001, 3)
    if shape == "pair":
        more = np.full((2, 900000), 0)
        more[1] = 99
    elif shape == "pairs":
        more = np.stack([rng.integers(0, 3, 900000), rng.integers(50, 53, 900000)])
    else:  # as many targets of degree one, next to one another in the order
        more = np.stack([np.full(900000, 12), 200000 + np.arange(900000)])
    v0, v1 = np.concatenate([v0, more[0]]), np.concatenate([v1, more[1]])
    order = rng.permutation(len(v0))
    _same_csr(G, v0[order], v1[order])


# bottom-up scans read a few entries past the last row: padding in either form
def test_search_after_the_general_sort(G):
    print("\n[general] search", flush=True)
    rng = np.random.default_rng(9)
    v0 = np.concatenate([np.full(200000, 3), rng.integers(0, 50000, 300000)]).astype(np.int64)
    v1 = np.concatenate([np.full(200000, 8), rng.integers(0, 50000, 300000)]).astype(np.int64)
    g = _same_csr(G, v0, v1)
    bfs = G.Bfs(g)
    for root in (3, int(v0[-1])):
        for alpha in (10.0, 1e9):
            bfs.run(root, 16, alpha, 14.0)
            ok, _, errs = bfs.validate(root)
            assert ok, errs
