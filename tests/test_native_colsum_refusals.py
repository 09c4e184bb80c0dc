"""What the entries for column sums, joint casts and weight gradients as stored refuse before they touch the GPU: null pointers, sizes off
their multiples, and column counts that leave no slab at all."""
import ctypes

import pytest

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


def test_null_pointers(L):
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
