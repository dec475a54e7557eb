"""Which kernel a call takes, and in which shape, is found once per size and not on every call (no GPU needed)."""
import ctypes
import time

import pytest

from modular_amd import _lib


def microseconds(call, calls=400, repeats=15):
    """of one call: the best of several rounds, each of many"""
    best = float("inf")
    for _ in range(repeats):
        start = time.perf_counter()
        for _ in range(calls):
            call()
        best = min(best, time.perf_counter() - start)
    return best / calls * 1e6


# (T, N, K, granularity): 17 to 2048 rows, where several kernels and many shapes are compared; a decode of one row is answered without any comparison
QKV = [(T, 6144, 4096, gran) for T in (20, 64, 200, 777, 2011) for gran in (_lib.GRAN_BLOCK, _lib.GRAN_ROWWISE)]


@pytest.mark.parametrize("size", QKV)
def test_fused_qkv_workspace(size):
    need = _lib.lib().maxfp8_linear_qkv_workspace_bytes
    assert microseconds(lambda: need(*size)) < 3 * microseconds(lambda: need(1, *size[1:])) + 0.3


@pytest.mark.parametrize("M", [20, 64, 117, 600, 1777])
@pytest.mark.parametrize("gran", [_lib.GRAN_BLOCK, _lib.GRAN_ROWWISE])
def test_linear_workspace(M, gran):
    need = _lib.lib().maxfp8_linear_workspace_bytes
    assert microseconds(lambda: need(M, 6144, 4096, gran)) < 3 * microseconds(lambda: need(1, 6144, 4096, gran)) + 0.3


def test_small_tiles_by_name():
    """the text of a small tile names its shape, which takes the same search as its launch"""
    text = ctypes.create_string_buffer(256)
    describe = lambda M: _lib.lib().maxfp8_matmul_describe(M, 6144, 4096, 1, 1, text, len(text))
    describe(117)
    assert b"per CU" in text.value
    # (the text itself takes a few tenths of a microsecond, the search 1 to 3)
    assert microseconds(lambda: describe(117)) < 2 * microseconds(lambda: describe(1)) + 0.3


def test_the_same_size_asked_in_different_ways():
    """answers of one kind of call are not those of another, nor of other tuning switches"""
    lib = _lib.lib()
    for _ in range(2):
        assert _lib.matmul_describe(48, 8192, 28672) != _lib.matmul_describe(48, 8192, 28672, True, False)
        assert lib.maxfp8_fused_qkv_matmul_workspace_bytes(512, 7168, 16384, 1) > 0
        assert lib.maxfp8_linear_workspace_bytes(117, 6144, 4096, _lib.GRAN_BLOCK) > 117 * 4096


def test_other_switches_other_answers(tune):
    plain = _lib.matmul_describe(117, 6144, 4096)
    tune(MAXFP8_MID="244")
    assert _lib.matmul_describe(117, 6144, 4096) != plain
    tune(MAXFP8_MID=None)
    assert _lib.matmul_describe(117, 6144, 4096) == plain
