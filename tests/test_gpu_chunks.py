"""Bottom-up levels over chunks of every size, at their edges, against the oracle."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import g500bfs
    g500bfs.load()
    return g500bfs


# chunks hold 8 to 64 bitmap words of 64 vertices: vertex counts around one
# chunk of 8 words, one word, and an odd number of words
@pytest.mark.parametrize("vertices", [3, 63, 64, 65, 511, 512, 513, 1025, 40001])
def test_bottom_up_at_chunk_edges(G, vertices):
    print(f"\n[chunks] {vertices} vertices", flush=True)
    rng = np.random.default_rng(vertices)
    # every vertex hangs on a random earlier one and on a few others
    v0 = np.arange(1, vertices, dtype=np.int64)
    v1 = (rng.random(vertices - 1) * v0).astype(np.int64)
    extra = rng.integers(0, vertices, (2, 3 * vertices))
    v0, v1 = np.concatenate([v0, extra[0]]), np.concatenate([v1, extra[1]])
    g = G.Graph.from_edges(v0, v1).construct()
    og = O.Graph(v0, v1)
    bfs = G.Bfs(g)
    for root in (0, int(v0[-1])):
        for alpha in (10.0, 1e9):  # 1e9: bottom-up from the second level on
            ref = og.bfs(root)
            bfs.run(root, 16, alpha, 14.0)
            lev = bfs.levels()
            assert np.array_equal(lev, np.where(ref < 0, 0xFFFF, ref).astype(np.uint16))
            ok, _, errs = bfs.validate(root)
            assert ok, errs


# more words than waves at 8 words a chunk, so chunks grow to 16, 32 and 64
@pytest.mark.parametrize("scale", [21, 23, 25])
def test_larger_chunks_validate(G, scale, golden):
    print(f"\n[chunks] scale {scale}", flush=True)
    g = G.Graph.generate(scale).construct()
    bfs = G.Bfs(g)
    for r in g.find_roots(3).tolist():
        for alpha in (10.0, 1e9):
            bfs.run(r, 16, alpha, 14.0)
            ok, te, errs = bfs.validate(r)
            assert ok and te == golden["pf_nedge"][scale], errs
