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


@pytest.mark.parametrize("x,N,M,K,code", [
    (F32, (4096,), 16, 512, 9), (F32, (2048,), 32, 512, 9), (F32, (2048,), 32, 1280, 9), (F32, (2048,), 32, 1296, 8), (F32, (2048,), 64, 512, 10),
    (F32, (4096,), 64, 1024, 11), (F32, (4096,), 65, 1024, None), (F32, (4096,), 64, 1040, None),
    (BF16, (1000,), 17, 1040, 9), (BF16, (2048,), 64, 512, 10), (BF16, (2048,), 64, 4096, None),
    (BF16, (2000, 48), 32, 256, 9), (BF16, (2000, 49), 32, 256, 10),
    (F32, (5120,), 3, 1536, 10), (BF16, (5120,), 3, 1536, 9), (BF16, (4096,), 3, 1536, 8)])
def test_tiles_of_16_rows_where_they_run_in_one_round(x, N, M, K, code):
    """Codes 8 to 11: 16 rows of X against 16, 16, 32 and 64 of W. Short rows of K were up to 1.4 times slower on the
    larger tiles than on the kernel before those."""
    form = _form(x, N, M, K, False)
    assert form < 8 if code is None else form == code


@pytest.mark.parametrize("M,N,K", [(2048, 5120, 1536), (2048, 5120, 2048), (1500, 4096, 1536)])
def test_many_rounds_are_not_left_to_the_form_without_k_groups(M, N, K):
    """Form 4 of the fp32 table: 110 us at the first size, the 256 x 256 tiles before it 97, form 6 80."""
    assert _form(F32, (N,), M, K, False) != 4
