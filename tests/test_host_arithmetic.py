"""Plain host code of the library (tests/cpp/host_checks.cpp), on the CPU."""
import ctypes
import os
import subprocess

import pytest

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")


@pytest.fixture(scope="module")
def lib():
    so = os.path.join(CPP, "libhost_checks.so")
    if not os.path.exists(so):
        subprocess.run(["make", "-C", CPP, "libhost_checks.so"], check=True)
    return ctypes.CDLL(so)


# sums of sizes and padding at and beyond 2^32
@pytest.mark.parametrize("align", [1, 8, 1 << 20])
@pytest.mark.parametrize("size", [[], [5], [1, 2, 3, 4], [600 << 20] * 4, [2 ** 32 - 1] * 4, [2 ** 32 - 1, 1, 2 ** 31]])
def test_places_of_objects(lib, size, align):
    at = (ctypes.c_uint64 * 4)()
    lib.host_place_run.restype = ctypes.c_uint64
    end = lib.host_place_run((ctypes.c_uint32 * 4)(*size), len(size), align, at)
    want = 0
    for k, s in enumerate(size):
        assert at[k] == want
        want += (s + align - 1) // align * align
    assert end == want


# bytes of a state's begin, size and magnitude buffers (0: no buffer), and the objects they hold
@pytest.mark.parametrize("bytes_of,objects", [((0, 0, 0), 0), ((0, 256, 256), 0), ((8, 256, 256), 0), ((256, 0, 256), 0),
                                              ((256, 256, 0), 0), ((24, 256, 256), 2), ((256, 256, 256), 16),
                                              ((1 << 40, 12, 1 << 40), 3), ((8 * 101, 400, 1600), 100)])
def test_room_of_a_state(lib, bytes_of, objects):
    lib.host_state_room.restype = ctypes.c_uint64
    assert lib.host_state_room(*map(ctypes.c_uint64, bytes_of)) == objects


# buffers that the pool keeps: those that the device is known to have finished
# with, of 64 KB to half its 4 GiB, the newest that fit
@pytest.mark.parametrize("n,failing,size,kept", [(1, 0, 1 << 20, 1), (1, 1, 1 << 20, 0), (5, 2, 1 << 20, 3),
                                                 (3, 0, 1 << 15, 0), (3, 0, 3 << 30, 0), (6, 0, 1 << 30, 4),
                                                 (70, 0, 1 << 20, 64)])
def test_pooled_buffers(lib, n, failing, size, kept):
    lib.host_pool_give.restype = ctypes.c_uint64
    freed = ctypes.c_uint64()
    assert lib.host_pool_give(*map(ctypes.c_uint64, (n, failing, size)), ctypes.byref(freed)) == kept * size
    assert freed.value == n - kept
