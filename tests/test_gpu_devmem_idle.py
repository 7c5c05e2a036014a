"""Device memory of freed graphs goes back without a call that allocates or asks for it."""
import ctypes as C
import time

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import g500bfs
    g500bfs.load()
    return g500bfs


def _free_bytes():
    """Free device memory as another user of the device sees it (nothing is given back)."""
    hip = C.CDLL("libamdhip64.so.7")  # the one the library runs on
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_idle_blocks_go_back_while_searching(G):
    print("\n[devmem] idle", flush=True)
    small = G.Graph.generate(12).construct()
    bfs, batch = G.Bfs(small), G.MultiBfs(small, max_roots=8)
    roots = small.find_roots(8)
    G.device_memory()
    for search in (lambda: bfs.run(int(roots[0])), lambda: batch.run(roots)):
        search()
        before = _free_bytes()
        big = G.Graph.generate(22).construct()
        big.free()
        kept = before - _free_bytes()
        assert kept > 512 << 20  # more than the edges alone
        search()
        assert before - _free_bytes() == kept
        time.sleep(10.5)
        search()
        assert before - _free_bytes() < 64 << 20
