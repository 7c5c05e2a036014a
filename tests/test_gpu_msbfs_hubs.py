"""Batched levels where hubs are pulled from, against the plain engine."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import g500bfs
    g500bfs.load()
    return g500bfs


@pytest.fixture(scope="module")
def s14(G):
    g = G.Graph.generate(14).construct()
    bfs = G.Bfs(g)
    roots = g.find_roots(256)
    levels = {}
    for r in roots.tolist():
        bfs.run(r)
        lv = bfs.levels()
        levels[r] = np.where(lv == 0xFFFF, 0xFF, lv).astype(np.uint8)
    return g, roots, levels


# one to four lane words, their ends, heavy bins from a few hubs to every
# vertex, top-down levels of any weight (td_alpha 1), split levels off, as
# usual and with every root pushing, rows in one and in many work items
@pytest.mark.parametrize("roots", [1, 64, 65, 128, 150, 256])
@pytest.mark.parametrize("tuning", [
    dict(heavy_degree=1024, medium_degree=64), dict(heavy_degree=64, medium_degree=8),
    dict(heavy_degree=1, medium_degree=1, heavy_chunk=256),
    dict(heavy_degree=256, medium_degree=16, heavy_chunk=256, td_alpha=1.0),
    dict(heavy_degree=64, medium_degree=8, split_bp=10000, td_alpha=50.0),
    dict(heavy_degree=64, medium_degree=8, split_bp=0, medium_group=4)])
def test_hub_pulls_keep_levels(G, s14, roots, tuning):
    print(f"\n[hubs] {roots} roots {tuning}", flush=True)
    g, all_roots, levels = s14
    mb = G.MultiBfs(g, max_roots=roots)
    mb.set_tuning(**tuning)
    r = all_roots[:roots]
    for _ in range(2):
        mb.run(r)
    for i in {0, roots // 2, roots - 1}:
        assert np.array_equal(mb.levels(i), levels[int(r[i])]), i
    mb.destroy()
