"""Device memory kept between allocations: given back when asked for, safe to reuse."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import g500bfs
    g500bfs.load()
    return g500bfs


def _levels(G, scale, seed, roots=2):
    g = G.Graph.generate(scale, 16, 2 + seed, 3 + seed).construct()
    b = G.Bfs(g)
    out = []
    for r in g.find_roots(roots).tolist():
        b.run(r)
        ok, _, errs = b.validate(r)
        assert ok, errs
        out.append(b.levels())
    b.destroy()
    g.free()
    return out


def test_freed_memory_is_given_back(G):
    print("\n[devmem] given back", flush=True)
    _levels(G, 16, 0)  # the runtime's own first-use memory
    before, total = G.device_memory()
    for seed in range(3):
        _levels(G, 20, seed)
    after, _ = G.device_memory()
    assert before - after < 64 << 20, (before, after, total)


# larger, then smaller graphs: their arrays lie in blocks that hold other data
def test_results_in_reused_blocks(G):
    print("\n[devmem] reuse", flush=True)
    fresh = {}
    for scale in (17, 18, 19):
        G.device_memory()  # gives the kept blocks back
        fresh[scale] = _levels(G, scale, 5)
    for scale in (19, 18, 17, 18, 19):
        for a, b in zip(_levels(G, scale, 5), fresh[scale]):
            assert np.array_equal(a, b)


def test_reuse_from_several_threads(G):
    print("\n[devmem] threads", flush=True)
    want = {s: _levels(G, 17, s) for s in range(3)}
    wrong = []

    def work(seed):
        for _ in range(3):
            got = _levels(G, 17, seed)
            if not all(np.array_equal(a, b) for a, b in zip(got, want[seed])):
                wrong.append(seed)

    ts = [threading.Thread(target=work, args=(s,)) for s in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong
