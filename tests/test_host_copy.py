"""gr_host_copy and the arrays that frames are delivered in (no GPU needed)."""
import os
import signal
import subprocess
import sys
import threading

import numpy as np
import pytest

from gorender_amd import _lib
from gorender_amd.device import ResultArrays

PIECE = 128 << 10
SHARED = 512 << 10


@pytest.mark.parametrize("n", [0, 1, PIECE, SHARED - 1, SHARED, SHARED + 1, 8 * PIECE + 3,
                               (9 << 20) + 5])
def test_host_copy(n):
    """Below and above the shared size, of whole and of broken pieces; nothing
    past the end is touched."""
    src = np.random.default_rng(n).integers(0, 256, n + 1, dtype=np.uint8)
    dst = np.zeros(n + 64, np.uint8)
    _lib.check(_lib.load().gr_host_copy(dst.ctypes.data, src.ctypes.data, n))
    assert np.array_equal(dst[:n], src[:n]) and not dst[n:].any()


def test_host_copy_refuses_null():
    with pytest.raises(_lib.GorenderError) as e:
        _lib.check(_lib.load().gr_host_copy(None, None, 1))
    assert e.value.status == _lib.GR_ERR_INVALID_ARGUMENT


def test_host_copy_from_several_threads():
    """Copies at once from four threads, most of which find the helpers taken."""
    lib = _lib.load()
    bad = []

    def work(seed):
        rng = np.random.default_rng(seed)
        for k in range(40):
            src = rng.integers(0, 256, SHARED + 1000 * k + seed, dtype=np.uint8)
            dst = np.zeros_like(src)
            _lib.check(lib.gr_host_copy(dst.ctypes.data, src.ctypes.data, src.nbytes))
            if not np.array_equal(src, dst):
                bad.append((seed, k))

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_result_arrays_reuse_only_what_is_free():
    pool = ResultArrays()
    a = pool.empty(np.float32, (512, 512))
    at = a.ctypes.data
    b = pool.empty(np.uint8, (512, 512, 4))
    assert b.ctypes.data != at
    view = a[100:]
    del a
    c = pool.empty(np.float32, (512, 512))
    assert c.ctypes.data not in (at, b.ctypes.data)  # a view is still in use
    del view
    d = pool.empty(np.float32, (1024, 256))
    assert d.ctypes.data == at and d.dtype == np.float32 and d.shape == (1024, 256)


def test_result_arrays_are_bounded():
    pool = ResultArrays()
    pool.LIMIT = 4 << 20
    held = [pool.empty(np.uint8, (1 << 20,)) for _ in range(6)]
    assert pool._bytes == 4 << 20
    assert len({h.ctypes.data for h in held}) == 6
    del held
    other = pool.empty(np.uint8, (3 << 20,))  # free blocks of another size make room
    assert pool._bytes == 3 << 20 and other.nbytes == 3 << 20
    assert pool.empty(np.uint8, (10,)).base is None  # small arrays are their own
    pool.clear()
    other[:] = 1


def test_result_arrays_do_not_rest_on_reference_counts(monkeypatch):
    """What an interpreter counts for a local or an argument is its own business:
    memory is on loan as long as an array or a view of it lives."""
    pool = ResultArrays()
    monkeypatch.setattr(sys, "getrefcount", lambda o: 3)
    held = [pool.empty(np.uint8, (512, 512, 4))[1:] for _ in range(4)]
    assert len({h.ctypes.data for h in held}) == 4
    for k, h in enumerate(held):
        h[:] = k
    assert [int(h.max()) for h in held] == [0, 1, 2, 3]


def test_result_arrays_from_several_threads():
    """Arrays taken, filled and dropped by four threads at once, a few kept across
    turns: none is handed out twice, and the blocks stay few."""
    pool = ResultArrays()
    bad = []

    def work(seed):
        kept = []
        for k in range(300):
            a = pool.empty(np.uint32, (256, 256 + 64 * (k % 3)))
            a[:] = seed * 1000 + k
            kept.append((seed * 1000 + k, a[5:]))
            if len(kept) == 4:
                v, a = kept.pop(k % 4)
                if not (a == v).all():
                    bad.append((seed, k))

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    pool.empty(np.uint8, (1 << 18,))
    assert pool._bytes <= 3 * 4 * 5 * (256 * 384 * 4)


def test_result_arrays_on_loan_outlive_a_cleared_pool():
    pool = ResultArrays()
    a = pool.empty(np.uint8, (1 << 20,))
    a[:] = 7
    pool.clear()
    b = pool.empty(np.uint8, (1 << 20,))
    b[:] = 9
    assert (a == 7).all()
    del a  # its memory goes: it is not the cleared pool's any more
    c = pool.empty(np.uint8, (1 << 20,))
    assert pool._bytes == 2 << 20
    assert c.ctypes.data != b.ctypes.data


def test_host_copy_in_a_forked_child():
    """The helper threads stay in the process that started them."""
    lib = _lib.load()
    src = np.random.default_rng(3).integers(0, 256, 8 << 20, dtype=np.uint8)
    dst = np.zeros_like(src)
    _lib.check(lib.gr_host_copy(dst.ctypes.data, src.ctypes.data, src.nbytes))
    pid = os.fork()
    if pid == 0:
        signal.alarm(20)
        dst[:] = 0
        ok = lib.gr_host_copy(dst.ctypes.data, src.ctypes.data, src.nbytes) == 0
        os._exit(0 if ok and np.array_equal(src, dst) else 1)
    assert os.waitpid(pid, 0)[1] == 0


def test_library_stays_while_its_threads_wait():
    """Closing the library leaves its code mapped: helper threads wait in it."""
    code = (
        "import _ctypes, ctypes, sys\n"
        "lib = ctypes.CDLL(sys.argv[1])\n"
        "a, b = ctypes.create_string_buffer(b'x' * (8 << 20)), ctypes.create_string_buffer(8 << 20)\n"
        "n = ctypes.c_size_t(8 << 20)\n"
        "assert lib.gr_host_copy(b, a, n) == 0 and b.raw[: 8 << 20] == a.raw[: 8 << 20]\n"
        "_ctypes.dlclose(lib._handle)\n"
        "assert sys.argv[1] in open('/proc/self/maps').read(), 'unmapped'\n"
        "again = ctypes.CDLL(sys.argv[1])\n"
        "ctypes.memset(b, 0, 8 << 20)\n"
        "assert again.gr_host_copy(b, a, n) == 0 and b.raw[: 8 << 20] == a.raw[: 8 << 20]\n")
    path = os.path.realpath(_lib.ALT_LIB_PATH or _lib.LIB_PATH)
    r = subprocess.run([sys.executable, "-c", code, path], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
