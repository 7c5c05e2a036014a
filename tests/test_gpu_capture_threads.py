"""Engines that capture their batches beside threads that build graphs and copy results."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import g500bfs
    g500bfs.load()
    return g500bfs


def test_captures_beside_builds(G):
    print("\n[capture] threads", flush=True)
    g = G.Graph.generate(16).construct()
    roots = g.find_roots(64)
    first = G.MultiBfs(g, max_roots=64)
    first.run(roots)
    te = first.te()
    level = [first.levels(i) for i in range(64)]
    wrong, stop = [], threading.Event()

    def build(seed):
        try:
            while not stop.is_set():
                h = G.Graph.generate(17, 16, 2 + seed, 3).construct()
                bfs = G.Bfs(h)
                root = int(h.find_roots(1)[0])
                bfs.run(root)
                ok, _, errs = bfs.validate(root)
                if not ok:
                    wrong.append(errs)
                bfs.levels()
                bfs.destroy()
                h.free()
        except G.G500Error as e:
            wrong.append(str(e))

    ts = [threading.Thread(target=build, args=(s,)) for s in range(2)]
    for t in ts:
        t.start()
    try:
        for i in range(40):
            batch = G.MultiBfs(g, max_roots=64)
            n = 20 + i
            for _ in range(3):  # the capture, then replays
                batch.run(roots[:n])
                assert np.array_equal(batch.te(), te[:n])
            assert np.array_equal(batch.levels(n - 1), level[n - 1])
            batch.destroy()
    finally:
        stop.set()
        for t in ts:
            t.join()
    assert not wrong, wrong[:3]


# a thread that only takes and frees device memory
def test_captures_beside_releases(G):
    print("\n[capture] releases", flush=True)
    g = G.Graph.generate(14).construct()
    roots = g.find_roots(8)
    first = G.MultiBfs(g, max_roots=8)
    first.run(roots)
    te = first.te()
    wrong, stop = [], threading.Event()

    def release():
        try:
            while not stop.is_set():
                G.Graph.create(1 << 20).free()
        except G.G500Error as e:
            wrong.append(str(e))

    t = threading.Thread(target=release)
    t.start()
    try:
        for i in range(40):
            batch = G.MultiBfs(g, max_roots=8)
            batch.run(roots)
            assert np.array_equal(batch.te(), te)
            batch.destroy()
    finally:
        stop.set()
        t.join()
    assert not wrong, wrong[:3]
