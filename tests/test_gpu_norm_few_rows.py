"""The norms' forward kernels in narrower blocks where there are few rows: the bits that the same rows have among many, and the maximum,
around the row counts where the block's width changes and for every width of a row."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("cols", [264, 768, 1024, 2048, 4096, 8192])
def test_a_row_has_the_same_bits_among_few_and_many(cols, dtype):
    from optimus_dl_amd import native as N

    many = 34000 if cols <= 2048 else 9000
    g = torch.Generator(device="cuda").manual_seed(cols)
    x = torch.randn((many, cols), device="cuda", generator=g).to(dtype)
    w, b = (torch.randn(cols, device="cuda", generator=g) for _ in range(2))
    rms, ln = N.rmsnorm_amax_parts(x, w, 1e-5), N.layernorm_amax_parts(x, w, b, 1e-5) if cols <= 4096 else None
    for rows in (1, 3, 67, 512, 1363, 2047, 2048, 2731, 4095, 4096, 5461, 8176, 8191, 8193):
        y, rstd, parts = N.rmsnorm_amax_parts(x[:rows], w, 1e-5)
        assert torch.equal(y, rms[0][:rows]) and torch.equal(rstd, rms[1][:rows]) and parts.numel() == N.AMAX_PARTS
        assert parts.max().item() == y.float().abs().max().item()
        if ln is not None:
            y, *stats, parts = N.layernorm_amax_parts(x[:rows], w, b, 1e-5)
            assert torch.equal(y, ln[0][:rows]) and all(torch.equal(s, l[:rows]) for s, l in zip(stats, ln[1:3], strict=True))
            assert parts.max().item() == y.float().abs().max().item()
