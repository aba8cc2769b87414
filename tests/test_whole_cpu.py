"""lasp_whole_ok and what lasp_whole_fwd refuses, without a GPU: every check comes before anything is launched."""
import ctypes

import pytest

from lasp_amd import _abi

P, MB = ctypes.c_void_p, 1 << 20


@pytest.fixture(scope="module")
def lib():
    return _abi.load()


def ok(lib, b, h, n, d, e, dtype=1, backward=1):
    return lib.lasp_whole_ok(b, h, ctypes.c_int64(n), d, e, dtype, backward)


def test_lines(lib):
    assert ok(lib, 2, 12, 2048, 128, 128) == 1 and ok(lib, 2, 12, 2048, 128, 128, 2) == 1
    assert ok(lib, 2, 12, 2113, 128, 128) == 0                                       # beyond 88 tokens per (b, h)
    assert ok(lib, 2, 12, 1024, 128, 128) == 0                                       # one launch by plan
    assert ok(lib, 2, 12, 2048, 128, 128, 0) == 0 and ok(lib, 2, 12, 2048, 64, 64) == 0 and ok(lib, 2, 12, 2048, 256, 128) == 0
    assert ok(lib, 1, 64, 4096, 128, 128) == 1 and ok(lib, 1, 64, 4097, 128, 128) == 0  # four segments gathered
    assert ok(lib, 1, 68, 4700, 128, 128) == 1
    assert ok(lib, 1, 120, 6144, 128, 128, 1, 0) == 1 and ok(lib, 1, 120, 6144, 128, 128) == 0  # whose backward takes three kernels
    assert ok(lib, 1, 24, 1920, 96, 96, 1, 0) == 1 and ok(lib, 1, 24, 1921, 96, 96, 1, 0) == 0  # narrow rows
    assert ok(lib, 1, 512, 6144, 128, 128, 1, 0) == 1 and ok(lib, 1, 512, 6145, 128, 128, 1, 0) == 0
    assert ok(lib, 2, 12, 2048, 128, 129) == 0 and ok(lib, 0, 12, 2048, 128, 128) < 0


def test_what_is_refused(lib):
    fwd = lib.lasp_whole_fwd
    fwd.restype = ctypes.c_int
    fwd.argtypes = [P] * 8 + [ctypes.c_int] * 2 + [ctypes.c_int64] + [ctypes.c_int] * 3 + [P]
    size = 24 * 128 * 128 * 4

    def call(n=2048, q=16 * MB, kv_in=None, kv_out=None, twin=None, dtype=1):
        return fwd(q, 32 * MB, 48 * MB, MB, kv_in, kv_out, twin, 64 * MB, 2, 12, n, 128, 128, dtype, None)

    assert call(n=4096) == -2 and b"lasp_whole_ok" in lib.lasp_last_error()
    assert call(dtype=0) == -2
    assert call(q=None) == -1
    assert call(kv_in=80 * MB, kv_out=80 * MB) == -8 and call(kv_in=80 * MB, kv_out=80 * MB + size - 4) == -8
    assert call(kv_in=80 * MB, kv_out=90 * MB, twin=90 * MB) == -8 and call(kv_in=80 * MB, twin=90 * MB) == -1
    assert call(q=16 * MB + 8) == -6 and call(kv_in=80 * MB + 2, kv_out=90 * MB) == -6
