"""The input of several Linears cast in one launch under delayed scaling (odl_fp8_cast_delayed_many): the codes and inverse scales of
separate casts, bit for bit, and their maxima, at the edges of tiles and with rows of padding behind x."""
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [O.E4M3, O.E5M2])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("count", [1, 2, 3, 4])
@pytest.mark.parametrize("rows,cols,rows_out", [(1, 8, 16), (16, 264, 16), (100, 1032, 128), (129, 64, 144), (1000, 1024, 1024), (560, 4096, 640)])
def test_codes_and_maxima_of_separate_casts(rows, cols, rows_out, count, dtype, fmt):
    from optimus_dl_amd import native as N

    x = (torch.randn((rows, cols), generator=torch.Generator().manual_seed(rows)) * 3).to(dtype).cuda()
    scales = [torch.tensor([s], device="cuda") for s in (0.5, 37.0, 1e4, 3e-3)[:count]]          # (the third saturates)
    strips = [[torch.zeros(N.AMAX_PARTS, device="cuda") for _ in scales] for _ in range(2)]
    strips[0][0][3] = strips[1][0][3] = 2.0 ** 40                                                  # of an earlier microbatch
    got = N.cast_delayed_many(x, scales, fmt, strips[0], rows_out)
    assert len(got) == count
    for (q, q_t, inv), s, own, other in zip(got, scales, strips[0], strips[1]):
        want = N.cast_delayed(x, s, fmt, other, want_transposed=True, rows_out=rows_out)
        assert torch.equal(q, want[0]) and torch.equal(q_t, want[1]) and torch.equal(inv, want[2]) and inv.shape == (1,)
        assert own.max().item() == other.max().item()


def test_what_one_launch_does_not_take_is_cast_one_by_one():
    from optimus_dl_amd import native as N

    for x in (torch.randn((33, 12), device="cuda"), torch.randn((16, 24), device="cuda")[:, 8:]):
        scale, parts = torch.ones(1, device="cuda"), [torch.zeros(N.AMAX_PARTS, device="cuda") for _ in range(3)]
        try:
            want = N.cast_delayed(x, scale, O.E4M3, parts[2], want_transposed=True, rows_out=48)
        except N.NativeError:
            with pytest.raises(N.NativeError):
                N.cast_delayed_many(x, [scale, scale], O.E4M3, parts[:2], 48)
            continue
        for got, own in zip(N.cast_delayed_many(x, [scale, scale], O.E4M3, parts[:2], 48), parts):
            assert all(torch.equal(a, b) for a, b in zip(got, want)) and own.max() == parts[2].max()


def test_nan_reaches_every_strip():
    from optimus_dl_amd import native as N

    x = torch.ones((32, 64), dtype=torch.bfloat16, device="cuda")
    x[5, 7] = float("nan")
    parts = [torch.zeros(N.AMAX_PARTS, device="cuda") for _ in range(2)]
    N.cast_delayed_many(x, [torch.ones(1, device="cuda")] * 2, O.E4M3, parts, 32)
    assert all(bool(p.isnan().any()) for p in parts)
