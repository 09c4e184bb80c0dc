"""What the entries for column sums, joint casts and weight gradients as stored refuse before they touch the GPU: null pointers, sizes off
their multiples, and column counts that leave no slab at all."""
import ctypes

import pytest
import torch

from optimus_dl_amd import native as N

P = 4096                                  # an address that is only looked at


@pytest.fixture(scope="module")
def L():
    if not N.is_built():
        pytest.skip("library not built")
    return N.load()


@pytest.mark.parametrize("src,cols,rows_out,fmt", [(1, 65544, 16, 0), (1, 131072, 16, 0), (0, 131080, 16, 0), (0, 12, 16, 0), (0, 16, 24, 0), (0, 16, 16, 7)])
def test_cast_with_sums(L, src, cols, rows_out, fmt):
    assert L.odl_fp8_cast_dynamic_colsum(P, src, 16, cols, rows_out, P, fmt, 0, P, P, P, P, P, 1, None) != 0


@pytest.mark.parametrize("src,rows,cols", [(0, 0, 16), (0, 16, 0), (0, 16, 12), (0, 16, 131080), (1, 16, 6), (1, 16, 65540), (2, 16, 16)])
def test_sums_of_slabs(L, src, rows, cols):
    assert L.odl_fp8_slabs_colsum(P, src, rows, cols, P, None) != 0


def test_null_pointers(L):
    assert L.odl_fp8_slabs_colsum(None, 0, 16, 16, P, None) != 0 and L.odl_fp8_slabs_colsum(P, 0, 16, 16, None, None) != 0
    for i in range(5):
        a = [P] * 5
        a[i] = None
        assert L.odl_fp8_gelu_bwd_slabs(a[0], a[1], 16, 16, P, a[2], a[3], a[4], None) != 0
    assert L.odl_fp8_gelu_bwd_slabs(P, P, 16, 12, P, P, P, P, None) != 0
    assert L.odl_fp8_amax_parts_slabs(P, 0, 16, 16, P, None, None) != 0
    assert L.odl_fp8_cast_dynamic_colsum(P, 0, 16, 16, 16, P, 0, 0, P, P, P, None, P, 1, None) != 0


@pytest.mark.parametrize("count,cols,rows_out", [(0, 16, 16), (5, 16, 16), (2, 12, 16), (2, 16, 24), (2, 16, 0)])
def test_joint_cast(L, count, cols, rows_out):
    arr = (ctypes.c_void_p * 5)(*[P] * 5)
    assert L.odl_fp8_cast_delayed_many(P, 0, 16, cols, rows_out, count, arr, 0, arr, arr, arr, arr, None) != 0


def test_joint_cast_null_member(L):
    full, hole = (ctypes.c_void_p * 2)(P, P), (ctypes.c_void_p * 2)(P, None)
    for i in range(5):
        a = [full] * 5
        a[i] = hole
        assert L.odl_fp8_cast_delayed_many(P, 0, 16, 16, 16, 2, a[0], 0, *a[1:], None) != 0


@pytest.mark.parametrize("n_out,n_in,tokens", [(240, 128, 512), (264, 128, 512), (272, 64, 512), (272, 128, 500), (272, 128, 384), (272, 128, 2**23), (0, 128, 512)])
def test_weight_gradient_as_stored(L, n_out, n_in, tokens):
    assert L.odl_fp8_gemm_wgrad(P, P, n_out, n_in, tokens, 1, 0, P, P, P, 1, None) != 0


@pytest.mark.parametrize("n_in,tokens", [(49152, 512), (50304, 512), (65536, 4096), (2**20, 512)])
def test_few_rows_of_a_wide_weight_are_not_sent_to_what_refuses_them(L, n_in, tokens):
    """Rows that leave no 256 x 256 tile, of so many columns that there are 192 tiles all the same."""
    for n_out in range(16, 256, 16):
        assert not N.gemm_wgrad_pays(n_out, n_in, tokens)
        assert L.odl_fp8_gemm_wgrad(P, P, n_out, n_in, tokens, 1, 0, P, P, P, 1, None) != 0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_what_pays_is_what_the_entry_takes(dtype):
    """The sizes of odl_fp8.h: n_out >= 256 in sixteens, n_in and tokens of 128, 512 tokens, operands and 264 rows of dW under 2 GiB."""
    taken = 0
    for n_out in (*range(8, 600, 8), 1040, 12304, 50304, 128 * 1024 + 16):
        for n_in in (64, 128, 700, 768, 4096, 25216, 50304, 2**20, 2**22):
            for tokens in (128, 384, 512, 520, 640, 8192, 2**15):
                if N.gemm_wgrad_pays(n_out, n_in, tokens, dtype):
                    taken += 1
                    assert n_out >= 256 and n_out % 16 == 0 and n_in % 128 == 0 and tokens % 128 == 0 and tokens >= 512
                    assert (n_out + 256) * tokens < 2**31 and (n_in + 256) * tokens < 2**31 and n_in * dtype.itemsize * 264 < 2**31
    assert taken > 10


@pytest.mark.parametrize("n_out,n_in", [(272, 50304), (528, 32768), (1040, 14336), (2064, 8192), (4112, 4096), (8208, 4096), (12304, 4096)])
def test_few_rows_keep_the_transposed_copy(n_out, n_in):
    """Faster over the copy, or not measured to be slower: no vocabulary's output."""
    assert not any(N.gemm_wgrad_pays(n_out, n_in, tokens, d) for tokens in (512, 2048, 8192) for d in (torch.bfloat16, torch.float32))
    assert N.gemm_wgrad_pays(12304, 3072, 2048) and N.gemm_wgrad_pays(32016, 5632, 8192)
