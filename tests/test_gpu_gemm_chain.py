"""Products that are added up in one launch (odl_fp8_gemm_nt_chain): the bits of a launch per product with the accumulate flag, at
sizes where tiles, rows and rounds of blocks end early."""
import ctypes

import pytest
import torch

from oracle import oracle as O
from tests.helpers import seeded_bf16

pytestmark = pytest.mark.gpu

WIDE, DEEP, DEEP192, TILED = 9, 10, 11, 4


@pytest.fixture(scope="module")
def N():
    from optimus_dl_amd import native

    native.load()
    native.init_device()
    return native


def forced(N, variant, call):
    N.gemm_set_variant(variant)
    try:
        return call()
    finally:
        N.gemm_set_variant(-1)


def make(M, cols, Ks, fmt_a, fmt_b, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    codes = lambda r, k, fmt: (torch.randn((r, k), device="cuda", generator=g) * 20).to(O.TORCH_FP8[fmt]).view(torch.uint8)
    scale = lambda i: torch.rand(1, device="cuda", generator=g) * 10.0 ** -i + 1e-3
    return ([codes(M, k, fmt_a) for k in Ks], [codes(cols, k, fmt_b) for k in Ks], [scale(i) for i in range(len(Ks))],
            [scale(1) for _ in Ks])


@pytest.mark.parametrize("variant", [WIDE, DEEP, DEEP192])
@pytest.mark.parametrize("M,cols,Ks", [(128, 128, (512, 512)), (130, 384, (768, 512)), (4016, 1152, (512, 1024, 512)), (257, 640, (1280, 512, 512, 768)),
                                       (8192, 2048, (512, 512)), (32, 128, (2048, 512))])
def test_chain_has_the_bits_of_accumulating_launches(N, M, cols, Ks, variant):
    a, b, sa, sb = make(M, cols, Ks, O.E5M2, O.E4M3, M + cols)
    want = forced(N, TILED, lambda: N.gemm_nt(a[0], b[0], O.E5M2, O.E4M3, sa[0], sb[0]))
    for s in range(1, len(Ks)):
        forced(N, TILED, lambda: N.gemm_nt(a[s], b[s], O.E5M2, O.E4M3, sa[s], sb[s], out=want, accumulate=True))
    got = forced(N, variant, lambda: N.gemm_nt_chain(a, b, O.E5M2, O.E4M3, sa, sb))
    assert got.dtype == torch.bfloat16 and torch.equal(got, want)


@pytest.mark.parametrize("fmt_a,fmt_b", [(O.E4M3, O.E4M3), (O.E5M2, O.E5M2)])
def test_chain_in_the_other_formats(N, fmt_a, fmt_b):
    a, b, sa, sb = make(300, 256, (512, 768), fmt_a, fmt_b, 1)
    got = forced(N, DEEP, lambda: N.gemm_nt_chain(a, b, fmt_a, fmt_b, sa, sb))
    want = N.gemm_nt(a[0], b[0], fmt_a, fmt_b, sa[0], sb[0])
    N.gemm_nt(a[1], b[1], fmt_a, fmt_b, sa[1], sb[1], out=want, accumulate=True)
    assert torch.equal(got, want)


def test_which_sums_run_in_one_launch(N):
    one = N.gemm_chain_in_one_launch
    assert one([3072, 3072], 8192, 1024) and one([5632, 5632], 4016, 2048) and one([1024, 512, 512], 1024, 1024)
    assert not one([14336, 14336], 8192, 4096) and not one([14336, 14336], 32, 4096)          # whole rounds; thin tiles
    assert not one([512, 256], 1024, 1024) and not one([640, 640], 1024, 1024) and not one([512, 512], 1024, 1000)
    assert not one([512], 1024, 1024) and not one([512] * 5, 1024, 1024) and not one([512, 512], 16, 1024)


def test_chain_refuses_what_does_not_fit(N):
    a, b, sa, sb = make(1024, 1024, (1024, 512), O.E5M2, O.E4M3, 2)
    with pytest.raises(N.NativeError):
        N.gemm_nt_chain(a, [b[0], b[1][:512]], O.E5M2, O.E4M3, sa, sb)
    with pytest.raises(N.NativeError):
        N.gemm_nt_chain(a, b, O.E5M2, O.E4M3, sa, [sb[0], sb[1].expand(2).contiguous()])
    with pytest.raises(N.NativeError):
        N.gemm_nt_chain(a, b, O.E4M3, O.E5M2, sa, sb)
    with pytest.raises(N.NativeError):                       # not faster, so there is no such launch
        x, y, p, q = make(64, 256, (512, 768), O.E5M2, O.E4M3, 2)
        N.gemm_nt_chain([t[:, :256].contiguous() for t in x], [t[:, :256].contiguous() for t in y], O.E5M2, O.E4M3, p, q)
    P, i64 = ctypes.c_void_p * 2, ctypes.c_int64 * 2
    p = lambda ts: P(*[t.data_ptr() for t in ts])
    rc = N.load().odl_fp8_gemm_nt_chain(2, p(a), p(b), i64(1024, 512), 1024, 1024, 1, 0, p(sa), None, a[0].data_ptr(), N._stream())
    assert rc != 0


@pytest.mark.parametrize("kind", ["tensorwise", "delayed", "mxfp8", "blockwise"])
@pytest.mark.parametrize("tokens", [1024, 4224])
def test_mlp_with_its_data_gradient_in_one_launch(N, monkeypatch, kind, tokens):
    """The bits of adding one by one.  Block scales have no such launch: the sum of two results, each rounded."""
    from optimus_dl_amd.modules import amp
    from optimus_dl_amd.modules.model.blocks import SwiGLUMLP
    from optimus_dl_amd.modules.model_transforms import build_model_transform

    def step(together):
        torch.manual_seed(3)
        mlp = build_model_transform({"_name": "fp8_linear"}).apply(SwiGLUMLP(2176 if kind == "mxfp8" else 2048, 1024).to("cuda", torch.bfloat16))
        kw = {"amax_history_len": 4} if kind == "delayed" else {}
        recipe = amp.create_fp8_recipe(kind, "hybrid", **kw)
        recipe.fuse_dgrad_gemm = together
        calls = []
        real = N.gemm_nt_chain
        monkeypatch.setattr(N, "gemm_nt_chain", lambda *args: (calls.append(1), real(*args))[1])
        x = seeded_bf16((tokens, mlp.w1.in_features), 1.0, 31).cuda().requires_grad_(True)
        with recipe.autocast():
            y = mlp(x)
        with recipe.backward():
            y.backward(seeded_bf16(tuple(y.shape), 1e-3, 32).cuda())
        monkeypatch.setattr(N, "gemm_nt_chain", real)
        return x.grad, [p.grad for p in mlp.parameters()], len(calls)

    (dx, dws, calls), (want, dws_want, none) = step(True), step(False)
    width = 2176 if kind == "mxfp8" else 2048
    block = kind in ("mxfp8", "blockwise")
    summed = not block and N.dgrad_sum_in_one_launch(tokens, width, [1024, 1024])
    assert none == 0 and calls == (0 if summed else int(not block and N.gemm_chain_in_one_launch([1024, 1024], tokens, width)))
    assert calls == 1 or tokens == 1024 or summed or block
    assert all(torch.equal(p, q) for p, q in zip(dws, dws_want))
    if not summed:
        assert torch.equal(dx, want)
    else:
        assert (dx.float() - want.float()).abs().max() <= 2.0 ** -7 * want.float().abs().max()


@pytest.mark.parametrize("kind", ["tensorwise", "delayed"])
def test_codes_of_the_data_gradient_are_gone_before_the_weight_gradients(N, monkeypatch, kind):
    """Both are one launch for gate and up, so the codes of both are there; those as stored are given back behind the first."""
    from optimus_dl_amd.modules import amp
    from optimus_dl_amd.modules.model.blocks import SwiGLUMLP
    from optimus_dl_amd.modules.model_transforms import build_model_transform

    mlp = build_model_transform({"_name": "fp8_linear"}).apply(SwiGLUMLP(1024, 3072).to("cuda", torch.bfloat16))
    recipe = amp.create_fp8_recipe(kind, "hybrid", amax_history_len=4)
    seen, chain, group = {}, N.gemm_nt_chain, N.gemm_nt_group

    def data_gradient(a, *args):
        dx = chain(a, *args)
        seen["codes"], seen["held"] = sum(t.numel() for t in a), torch.cuda.memory_allocated()
        return dx

    def products(a, b, fmt_a, *args):
        if fmt_a == O.E5M2:
            seen["left"] = torch.cuda.memory_allocated()
        return group(a, b, fmt_a, *args)

    monkeypatch.setattr(N, "gemm_nt_chain", data_gradient)
    monkeypatch.setattr(N, "gemm_nt_group", products)
    x = seeded_bf16((1024, 1024), 1.0, 31).cuda().requires_grad_(True)
    with recipe.autocast():
        y = mlp(x)
    with recipe.backward():
        y.backward(seeded_bf16(tuple(y.shape), 1e-3, 32).cuda())
    assert seen["codes"] == 2 * 1024 * 3072 and seen["left"] <= seen["held"] - seen["codes"]
