"""Weight gradients that read dY as stored where its columns are no whole tiles (odl_fp8_gemm_wgrad): the last tile begins before the end of
the one in front of it."""
import pytest
import torch
import torch.nn as nn

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n_out,n_in,tokens", [(256, 128, 512), (272, 128, 640), (496, 384, 512), (528, 256, 1152), (12304, 1024, 640), (50304, 768, 1024)])
def test_weight_gradient_of_rows_that_are_no_whole_tiles(n_out, n_in, tokens, out_dtype):
    """Against the tiled kernel over the transposed copy, which walks K in the same order; what lies behind each operand is NaN, and
    nothing in front of or behind the output is written."""
    from optimus_dl_amd import native as N

    g = torch.Generator(device="cuda").manual_seed(n_out + tokens)
    one = torch.tensor([0.25], device="cuda"), torch.tensor([0.5], device="cuda")

    def codes(r, c, fmt, nan):
        room = torch.full((r + 4, c), nan, dtype=torch.uint8, device="cuda")
        room[:r] = torch.randn((r, c), device="cuda", generator=g).to(O.TORCH_FP8[fmt]).view(torch.uint8)
        return room[:r]

    gy, x_t = codes(tokens, n_out, O.E5M2, 0x7E), codes(n_in, tokens, O.E4M3, 0x7F)
    N.gemm_set_variant(2)
    try:
        want = N.gemm_nt(gy.t().contiguous(), x_t, O.E5M2, O.E4M3, *one, out_dtype=out_dtype)
    finally:
        N.gemm_set_variant(-1)
    assert torch.equal(N.gemm_wgrad(gy, x_t, O.E5M2, O.E4M3, *one, out_dtype), want)

    room = torch.full((n_out + 512, n_in), 3.0, dtype=out_dtype, device="cuda")           # 256 rows each side: a tile's
    dw = room[256:256 + n_out]
    assert N.load().odl_fp8_gemm_wgrad(gy.data_ptr(), x_t.data_ptr(), n_out, n_in, tokens, O.E5M2, O.E4M3, one[0].data_ptr(), one[1].data_ptr(),
                                       dw.data_ptr(), N._OUT_DTYPES[out_dtype], N._stream()) == 0
    assert torch.equal(dw, want) and bool((room[:256] == 3.0).all()) and bool((room[256 + n_out:] == 3.0).all())


def test_weight_gradient_refusals():
    from optimus_dl_amd import native as N

    one = torch.ones(1, device="cuda")
    z = lambda r, c: torch.zeros((r, c), dtype=torch.uint8, device="cuda")
    for n_out, n_in, tokens in ((240, 128, 512), (264, 128, 512), (256, 64, 512), (256, 128, 576), (256, 128, 384)):
        with pytest.raises(N.NativeError):
            N.gemm_wgrad(z(tokens, n_out), z(n_in, tokens), O.E5M2, O.E4M3, one, one)
    assert N.gemm_wgrad_pays(50304, 768, 8192) and not N.gemm_wgrad_pays(50176, 768, 8192) and not N.gemm_wgrad_pays(1040, 768, 8192)
    assert not N.gemm_wgrad_pays(50304, 768, 8200) and not N.gemm_wgrad_pays(50304, 700, 8192)


@pytest.mark.parametrize("recipe_name", ["tensorwise", "delayed"])
def test_a_linear_takes_it_with_the_bits_of_the_copy(monkeypatch, recipe_name):
    from optimus_dl_amd import native as N
    from optimus_dl_amd.modules import amp
    from optimus_dl_amd.modules.fp8_linear import FP8Linear

    M, K, n_out = 496, 1024, 12304              # 49 x 4 tiles; the tokens are padded to 512
    x, dy = torch.randn((M, K), device="cuda").bfloat16(), (torch.randn((M, n_out), device="cuda") * 1e-3).bfloat16()
    lin = FP8Linear.from_linear(nn.Linear(K, n_out, bias=False).cuda())
    calls, real, grads = [], N.gemm_wgrad, []
    monkeypatch.setattr(N, "gemm_wgrad", lambda *a, **k: (calls.append(1), real(*a, **k))[1])
    for direct in ("auto", False):
        recipe = amp.create_fp8_recipe(recipe_name, "hybrid", amax_history_len=4)
        recipe.direct_layouts = direct
        for _ in range(2):                      # (delayed scaling: the second step runs on measured scales)
            lin.weight.grad = None
            with recipe.autocast():
                y = lin(x)
            with recipe.backward():
                y.backward(dy)
        grads.append(lin.weight.grad)
    assert len(calls) == 2 and torch.equal(*grads) and grads[0].dtype == torch.float32


@pytest.mark.parametrize("recipe_name", ["tensorwise", "delayed"])
@pytest.mark.parametrize("n_out", [128, 240])
def test_few_rows_of_a_wide_weight_keep_the_copy(n_out, recipe_name):
    """50304 -> 128: 197 tiles of 256 x 256, but not a whole one of rows."""
    from optimus_dl_amd.modules import amp
    from optimus_dl_amd.modules.fp8_linear import FP8Linear

    x, dy = torch.randn((512, 50304), device="cuda").bfloat16(), (torch.randn((512, n_out), device="cuda") * 1e-3).bfloat16()
    lin = FP8Linear.from_linear(nn.Linear(50304, n_out, bias=False).cuda().bfloat16())
    grads = []
    for direct in ("auto", False):
        recipe = amp.create_fp8_recipe(recipe_name, "hybrid", amax_history_len=4)
        recipe.direct_layouts = direct
        for _ in range(2):
            lin.weight.grad = None
            with recipe.autocast():
                y = lin(x)
            with recipe.backward():
                y.backward(dy)
        grads.append(lin.weight.grad)
    assert torch.equal(*grads) and bool(grads[0].any())
