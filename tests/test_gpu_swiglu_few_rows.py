"""Gate, up and their product of a few rows in one launch (odl_fp8_gemm_swiglu): every tile of its kernel, and sizes where rows, the
eight columns of a tile, the tiles of a block and the waves' shares of K end early, against the thin kernel's products and the
SwiGLU kernel, bit for bit."""
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu

THIN = 8


# (the SwiGLU kernel takes whole vectors of eight)
SIZES = [(r, c) for r in (1, 8, 16, 17, 32, 33, 64) for c in (4, 8, 12, 24, 1032, 3072, 5640, 8192, 10240, 14336, 16384) if r * c % 8 == 0]


@pytest.mark.parametrize("rows,cols", SIZES)
@pytest.mark.parametrize("K", [128, 1152, 4096])
def test_one_launch_has_the_bits_of_three(rows, cols, K):
    from optimus_dl_amd import native as N

    g = torch.Generator(device="cuda").manual_seed(rows + cols + K)
    codes = lambda r: (torch.randn((r, K), device="cuda", generator=g) * 20).to(O.TORCH_FP8[O.E4M3]).view(torch.uint8)
    x, gate, up = codes(rows), codes(cols), codes(cols)
    s = [torch.rand(1, device="cuda", generator=g) * 1e-2 for _ in range(3)]
    h, parts = N.gemm_swiglu(x, gate, up, O.E4M3, O.E4M3, *s)
    N.gemm_set_variant(THIN)
    try:
        a, b = N.gemm_nt(x, gate, O.E4M3, O.E4M3, s[0], s[1]), N.gemm_nt(x, up, O.E4M3, O.E4M3, s[0], s[2])
    finally:
        N.gemm_set_variant(-1)
    want, want_parts = N.swiglu_amax_parts(a.reshape(-1), b.reshape(-1))
    assert h.shape == (rows, cols) and torch.equal(h.reshape(-1), want)
    assert parts.numel() == N.AMAX_PARTS and parts.max().item() == want_parts.max().item()
