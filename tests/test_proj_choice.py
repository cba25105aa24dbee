"""Which tiles a projection of several weights takes (csrc/gemm_mid.hip, run on the host): the 256 x 256 tiles
run weights that they cannot stack one after the other, each in rounds of its own."""
import ctypes

import pytest

from aegist_mixer._lib import BF16, F32, lib


def _form(x_dtype, N, M, K, stacked):
    fn = getattr(lib(), "_ZN6aegist13gemm_mid_formEiiPKiiibb")
    fn.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_bool, ctypes.c_bool]
    arr = (ctypes.c_int * len(N))(*N)
    return fn(x_dtype, len(N), ctypes.cast(arr, ctypes.c_void_p), M, K, True, stacked)


@pytest.mark.parametrize("M", [1024, 1536])
def test_narrow_weights_that_are_not_stacked_count_their_own_rounds(M):
    assert _form(BF16, (8192, 4096, 32, 32), M, 2048, False) >= 0
    assert _form(BF16, (8192, 4096, 32, 32), M, 2048, True) == -1


def test_one_weight_is_a_stack_of_one():
    for x in (BF16, F32):
        for M in (65, 300, 1024, 4000, 20000):
            for N in (32, 512, 8192, 32768):
                assert _form(x, (N,), M, 2048, False) == _form(x, (N,), M, 2048, True)
