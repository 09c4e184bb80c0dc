"""Column sums on the way to a cast (odl_fp8_amax_parts_slabs, odl_fp8_gelu_bwd_slabs, odl_fp8_cast_dynamic_colsum, odl_fp8_slabs_colsum): the
codes, the scale and the sums are those of the separate launches, bit for bit, at the edges of tiles, slabs and column blocks."""
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(1, 8, 16), (16, 16, 16), (33, 264, 48), (320, 768, 320), (500, 1032, 640), (1000, 3072, 1024), (16400, 256, 16512), (40, 131072, 48)]


def parts_max(parts):
    return parts.max().reshape(1)


@pytest.mark.parametrize("fmt", [O.E4M3, O.E5M2])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,cols,rows_out", SHAPES)
def test_sums_finished_by_the_cast(rows, cols, rows_out, dtype, fmt):
    from optimus_dl_amd import native as N

    x = torch.randn((rows, cols), generator=torch.Generator().manual_seed(rows + cols)).to(dtype).cuda()
    if not N.colsum_supported(x):
        pytest.skip("more columns than the pass takes in fp32")
    want_parts, want_sums = N.amax_parts_colsum(x)
    want_q, want_qt, _, _, want_inv = N.cast_dynamic(x, want_parts, fmt, 1, rows_out=rows_out)
    for out in (torch.bfloat16, torch.float32):
        parts, slabs = N.amax_parts_colsum(x, finish=False)
        assert slabs.dim() == 2 and torch.equal(parts, want_parts)
        q, qt, inv, sums = N.cast_dynamic_colsum(x, parts, slabs, fmt, 1, rows_out, out)
        assert sums.dtype == out and torch.equal(sums, want_sums.to(out))
        assert torch.equal(inv, want_inv) and torch.equal(qt, want_qt) and torch.equal(q, want_q)


def test_sums_of_infinities_and_nan():
    from optimus_dl_amd import native as N

    x = torch.zeros((64, 32), dtype=torch.bfloat16)
    x[3, 1], x[5, 2], x[6, 2], x[9, 4] = float("inf"), float("inf"), float("-inf"), float("nan")
    x = x.cuda()
    _, want = N.amax_parts_colsum(x)
    parts, slabs = N.amax_parts_colsum(x, finish=False)
    sums = N.cast_dynamic_colsum(x, parts, slabs, O.E5M2, 0, 64, torch.bfloat16)[3]
    assert torch.equal(sums.isnan(), want.isnan()) and torch.equal(sums.nan_to_num(), want.to(torch.bfloat16).nan_to_num())
    assert sums[1].item() == float("inf") and bool(sums[2].isnan()) and bool(sums[4].isnan())


def test_columns_the_cast_does_not_take_are_finished_by_the_pass():
    from optimus_dl_amd import native as N

    x = torch.randn((48, 12), device="cuda")          # fp32: the pass takes multiples of four, the cast of eight
    want = N.amax_parts_colsum(x)
    got = N.amax_parts_colsum(x, finish=False)
    assert got[1].dim() == 1 and all(torch.equal(a, b) for a, b in zip(got, want))
    with pytest.raises(N.NativeError):
        N.cast_dynamic_colsum(x, *got, O.E4M3, 0, 48, torch.float32)


@pytest.mark.parametrize("rows,cols", [(r, c) for r, c, _ in SHAPES])
def test_gelu_backward_leaves_the_slabs(rows, cols):
    from optimus_dl_amd import native as N

    g = torch.Generator().manual_seed(rows * cols)
    x, dy = ((torch.randn((rows, cols), generator=g) * s).to(torch.bfloat16).cuda() for s in (2.0, 1e-2))
    want, want_parts = N.gelu_bwd_amax_parts(dy, x)
    dx, parts, slabs = N.gelu_bwd_slabs(dy, x)
    assert torch.equal(dx, want) and torch.equal(parts_max(parts), parts_max(want_parts))
    own_parts, own = N.amax_parts_colsum(dx, finish=False)
    used = (-(-rows // max(32, -(-(-(-rows // (N.AMAX_PARTS // -(-cols // 256)))) // 32) * 32))) * cols      # slabs x columns
    assert torch.equal(slabs.reshape(-1)[:used], own.reshape(-1)[:used])
    assert N.amax_parts_colsum(dx, finish=False, left=(parts, slabs))[1] is slabs


def test_slabs_are_not_handed_to_a_view_of_other_columns():
    from optimus_dl_amd.modules import amp

    recipe = amp.FP8Recipe(recipe_type="tensorwise")
    t = torch.zeros((64, 32), dtype=torch.bfloat16, device="cuda")
    parts, slabs = torch.zeros(4, device="cuda"), torch.zeros((2, 2), device="cuda")
    recipe.offer_parts(t, parts, slabs)
    assert recipe.take_parts_and_slabs(t.view(32, 64)) == (parts, None)
    recipe.offer_parts(t.view(2, 32, 32), parts, slabs)
    got = recipe.take_parts_and_slabs(t)
    assert got[0] is parts and got[1] is slabs


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [16, 16384, 48016])
def test_small_tensor_quantised_in_its_own_place(n, dtype):
    """Codes over the first bytes of x: the launch of one block, which reads everything first."""
    from optimus_dl_amd import native as N

    x = torch.randn((1, n), device="cuda").to(dtype)
    want, _, _, _, inv = N.quantise_small(x, O.E4M3)
    dyn, L = torch.empty(3, device="cuda"), N.load()
    assert L.odl_fp8_quantise_small(x.data_ptr(), 0 if dtype == torch.bfloat16 else 1, n, O.E4M3, 0, x.data_ptr(), dyn.data_ptr(), N._stream()) == 0
    assert torch.equal(x.view(torch.uint8).reshape(-1)[:n], want.reshape(-1)) and dyn[2].item() == inv.item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,cols", [(r, c) for r, c, _ in SHAPES])
def test_sums_finished_by_themselves(rows, cols, dtype):
    from optimus_dl_amd import native as N

    x = torch.randn((rows, cols), generator=torch.Generator().manual_seed(rows + 2 * cols)).to(dtype).cuda()
    if not N.colsum_supported(x):
        pytest.skip("more columns than the pass takes in fp32")
    _, want = N.amax_parts_colsum(x)
    left = N.amax_parts_colsum(x, finish=False)
    parts, sums = N.amax_parts_colsum(x, left=left)
    assert parts is left[0] and sums.shape == (cols,) and sums.dtype == torch.float32 and torch.equal(sums, want)
    with pytest.raises(N.NativeError):
        N.amax_parts_colsum(x, left=(parts, left[1][:1]))


@pytest.mark.parametrize("how", ["as stored", "both layouts", "frozen weight", "frozen weight and input", "wgrad off", "no bias", "bf16 Linear"])
def test_gelu_backward_makes_sums_where_they_are_used(monkeypatch, how):
    """c_fc behind its GELU: the slabs are made where c_fc has a bias and quantises its gradient or sums it, and used whichever layouts its
    cast writes; the gradients have the bits they have without them."""
    from optimus_dl_amd import native as N
    from optimus_dl_amd.modules import amp, fused
    from optimus_dl_amd.modules.model.blocks import GELUMLP
    from optimus_dl_amd.modules.model_transforms import build_model_transform

    n_in, n_out = (2048, 8192) if how == "as stored" else (256, 1024)
    torch.manual_seed(0)
    m = build_model_transform({"_name": "fp8_linear"}).apply(GELUMLP(n_in, n_out, bias=how != "no bias").to("cuda", torch.bfloat16))
    m.c_fc.weight.requires_grad_(not how.startswith("frozen"))
    m.c_fc.fp8_enabled = how != "bf16 Linear"
    recipe = amp.FP8Recipe(recipe_type="tensorwise", wgrad=how != "wgrad off")
    slabs_of, passes = [], []
    real_slabs, real_pass = N.gelu_bwd_slabs, N.amax_parts_colsum

    def counted(x, *a, left=None, **k):
        if left is None:
            passes.append(tuple(x.shape))
        return real_pass(x, *a, left=left, **k)

    monkeypatch.setattr(N, "gelu_bwd_slabs", lambda *a: (slabs_of.append(1), real_slabs(*a))[1])
    monkeypatch.setattr(N, "amax_parts_colsum", counted)

    def step():
        x = (torch.randn((4, 96, n_in), generator=torch.Generator().manual_seed(5))).bfloat16().cuda().requires_grad_("input" not in how)
        dy = (torch.randn((4, 96, n_in), generator=torch.Generator().manual_seed(6)) * 1e-2).bfloat16().cuda()
        for p in m.parameters():
            p.grad = None
        slabs_of.clear(); passes.clear()
        with recipe.autocast(), torch.autocast("cuda", torch.bfloat16):
            y = m(x)
        with recipe.backward():
            y.backward(dy)
        return [x.grad, *(p.grad for p in m.parameters())], len(slabs_of), passes.count((384, n_out))

    got, made, read_again = step()
    used = how not in ("no bias", "bf16 Linear")
    assert made == int(used) and read_again == 0
    monkeypatch.setattr(fused, "_gradient_is_summed", lambda x, recipe: False)
    want, made, read_again = step()
    assert made == 0 and read_again == int(used)
    assert all(a is b is None or torch.equal(a, b) for a, b in zip(got, want, strict=True))
