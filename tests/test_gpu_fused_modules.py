"""GPU: the fused SwiGLU / RMSNorm forwards inside real module trees.  What must hold:
the hand-over of partial maxima changes no bit (same codes, same outputs as the amax pass it
replaces), the amax passes it replaces are really gone, and the fused modules agree with the
modules' own PyTorch forwards to within a bf16 unit here and there (GEMM tolerance downstream)."""
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from oracle import oracle as O
from tests.helpers import max_rel_err, seeded_bf16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amp():
    from optimus_dl_amd.modules import amp as A

    return A


def make_mlp(n_embd=256, hidden=512, fuse=True, seed=0):
    from optimus_dl_amd.modules.model.blocks import SwiGLUMLP
    from optimus_dl_amd.modules.model_transforms import build_model_transform

    torch.manual_seed(seed)
    mlp = SwiGLUMLP(n_embd, hidden).to("cuda", torch.bfloat16)
    t = build_model_transform({"_name": "fp8_linear", "fuse_swiglu": fuse})
    t.apply(mlp)
    return mlp, t


def step(module, recipe, x, dy):
    xd = x.clone().requires_grad_(True)
    for p in module.parameters():
        p.grad = None
    with recipe.autocast():
        y = module(xd)
    with recipe.backward():
        y.backward(dy)
    return [y.detach(), xd.grad.detach()] + [p.grad.detach().clone() for p in module.parameters()]


def count_calls(monkeypatch, native, name):
    calls = []
    orig = getattr(native, name)

    def counted(*a, **kw):
        calls.append(tuple(a[0].shape))
        return orig(*a, **kw)

    monkeypatch.setattr(native, name, counted)
    return calls


def test_fused_mlp_skips_three_amax_passes_and_changes_no_bit(amp, monkeypatch):
    from optimus_dl_amd import native

    M, C, H = 384, 256, 512
    x = seeded_bf16((M, C), 1.0, 1).cuda()
    dy = seeded_bf16((M, C), 1e-3, 2).cuda()
    mlp, t = make_mlp(C, H, fuse=True)
    assert t.last_replacements.get("SwiGLU") == 1
    recipe = amp.FP8Recipe(recipe_type="tensorwise")
    amax_calls = count_calls(monkeypatch, native, "amax_parts")
    fused = step(mlp, recipe, x, dy)
    # x (shared by w1/w2), three weights, dy of c_proj: h, d_gate and d_up come with their maxima
    assert sorted(amax_calls) == sorted([(M, C), (H, C), (H, C), (C, H), (M, C)])
    assert recipe.producer_parts == []                                   # all three were taken
    # same modules, hand-over switched off: every tensor gets its own amax pass, results identical
    monkeypatch.setattr(type(recipe), "offer_parts", lambda self, t_, p_: None)
    amax_calls.clear()
    plain = step(mlp, recipe, x, dy)
    # the weights' codes are cached (unchanged Parameters): x, h, dy and the two gradients remain
    assert sorted(amax_calls) == sorted([(M, C), (M, H), (M, C), (M, H), (M, H)])
    for a, b in zip(fused, plain):
        assert torch.equal(a, b)


def test_fused_mlp_agrees_with_the_eager_activation(amp):
    M, C, H = 512, 256, 768
    x = seeded_bf16((M, C), 1.0, 3).cuda()
    dy = seeded_bf16((M, C), 1e-3, 4).cuda()
    fused_mlp, _ = make_mlp(C, H, fuse=True, seed=5)
    eager_mlp, t = make_mlp(C, H, fuse=False, seed=5)
    assert "SwiGLU" not in t.last_replacements
    recipe = amp.FP8Recipe(recipe_type="tensorwise")
    got = step(fused_mlp, recipe, x, dy)
    want = step(eager_mlp, recipe, x, dy)
    for name, a, b in zip(["y", "dx", "dw1", "dw2", "dwc"], got, want):
        assert max_rel_err(a, b) <= 1e-2, name


def test_swiglu_function_matches_torch_autograd(amp):
    from optimus_dl_amd.modules.fused import swiglu

    g = seeded_bf16((64, 256), 1.5, 6).cuda().requires_grad_(True)
    u = seeded_bf16((64, 256), 1.0, 7).cuda().requires_grad_(True)
    dh = seeded_bf16((64, 256), 1e-2, 8).cuda()
    recipe = amp.FP8Recipe(recipe_type="tensorwise")
    with recipe.autocast():
        h = swiglu(g, u)
    h.backward(dh)
    gc, uc, dhc = g.detach().cpu(), u.detach().cpu(), dh.cpu()
    assert torch.equal(h.detach().cpu().view(torch.int16), O.c_swiglu_fwd(gc, uc).view(torch.int16))
    wg, wu = O.c_swiglu_bwd(dhc, gc, uc)
    assert torch.equal(g.grad.cpu().view(torch.int16), wg.view(torch.int16))
    assert torch.equal(u.grad.cpu().view(torch.int16), wu.view(torch.int16))
    # outside a recipe: plain PyTorch
    h2 = swiglu(g.detach(), u.detach())
    assert torch.equal(h2, F.silu(g.detach()) * u.detach())


@pytest.mark.parametrize("in_dtype", [torch.float32, torch.bfloat16])
def test_fused_rmsnorm_feeds_the_linear_and_backpropagates(amp, monkeypatch, in_dtype):
    from optimus_dl_amd import native
    from optimus_dl_amd.modules.model.blocks import RMSNorm
    from optimus_dl_amd.modules.model_transforms import build_model_transform

    class Pre(nn.Module):
        def __init__(self):
            super().__init__()
            self.ln = RMSNorm(256, 1e-5)
            self.wq = nn.Linear(256, 320, bias=False)
            self.wk = nn.Linear(256, 128, bias=False)

        def forward(self, x):
            n = self.ln(x)
            return self.wq(n).float().sum(-1) + self.wk(n).float().sum(-1)

    torch.manual_seed(0)
    net = Pre().cuda()
    with torch.no_grad():
        net.ln.weight.copy_(torch.linspace(0.5, 1.5, 256))
    ref = Pre().cuda()
    ref.load_state_dict(net.state_dict())
    t = build_model_transform({"_name": "transformer_engine"})
    t.apply(net)
    assert t.last_replacements["RMSNorm"] == 1 and t.last_replacements["Linear"] == 2
    build_model_transform({"_name": "transformer_engine", "replace_norm": False}).apply(ref)
    x = (torch.randn(4, 96, 256, generator=torch.Generator().manual_seed(1)) * 2).to(in_dtype).cuda()
    recipe = amp.FP8Recipe(recipe_type="tensorwise")
    amax_calls = count_calls(monkeypatch, native, "amax_parts")
    outs = {}
    for name, m in (("fused", net), ("plain", ref)):
        xd = x.clone().requires_grad_(True)
        amax_calls.clear()
        with amp.fp8_autocast(torch.device("cuda"), recipe):
            y = m(xd)
        with amp.fp8_backward(recipe):
            y.sum().backward()
        outs[name] = (y.detach(), xd.grad.detach(), m.ln.weight.grad.detach(), m.wq.weight.grad.detach())
        if name == "fused":
            # the normalised activation arrives with its maxima: only the two weights and the two dy
            assert sorted(amax_calls) == sorted([(320, 256), (128, 256), (384, 320), (384, 128)])
        else:
            assert (4 * 96, 256) in amax_calls
    f, p = outs["fused"], outs["plain"]
    assert f[1].dtype == in_dtype
    assert max_rel_err(f[0], p[0]) <= 1e-2
    assert max_rel_err(f[1], p[1]) <= 2e-2
    assert max_rel_err(f[2], p[2]) <= 2e-2
    assert max_rel_err(f[3], p[3]) <= 1e-2


def test_fused_rmsnorm_equals_oracle_and_leaves_other_cases_alone(amp):
    from optimus_dl_amd.modules.fused import fuse_rmsnorm
    from optimus_dl_amd.modules.model.blocks import RMSNorm

    norm = RMSNorm(512, 1e-6).cuda()
    with torch.no_grad():
        norm.weight.copy_(torch.linspace(0.25, 2.0, 512))
    assert fuse_rmsnorm(norm) and not fuse_rmsnorm(norm)
    x = seeded_bf16((3, 40, 512), 3.0, 9)
    recipe = amp.FP8Recipe(recipe_type="tensorwise")
    with amp.fp8_autocast(torch.device("cuda"), recipe):
        y = norm(x.cuda())
        y32 = norm(x.float().cuda())                     # fp32 in, bf16 out under the bf16 autocast
    want, _ = O.c_rmsnorm(x, norm.weight.detach().cpu(), 1e-6)
    assert y.dtype == torch.bfloat16 and torch.equal(y.cpu().view(torch.int16), want.view(torch.int16))
    assert y32.dtype == torch.bfloat16 and torch.equal(y32.cpu().view(torch.int16), want.view(torch.int16))
    # no recipe: the module's own forward, dtype of the input
    y_plain = norm(x.float().cuda())
    assert y_plain.dtype == torch.float32
    # a recipe without the bf16 autocast around it and an fp32 input: own forward as well
    with recipe.autocast():
        assert norm(x.float().cuda()).dtype == torch.float32
        assert norm(x.cuda()).dtype == torch.bfloat16


@pytest.mark.parametrize("recipe_name", ["tensorwise", "delayed", "rowwise"])
def test_llama_block_with_fusions_trains_like_the_unfused_one(amp, recipe_name):
    from optimus_dl_amd.modules.model import Llama, LlamaConfig
    from optimus_dl_amd.modules.model_transforms import build_model_transform

    def build(fuse):
        torch.manual_seed(0)
        m = Llama(LlamaConfig(vocab_size=256, n_layer=2, n_head=4, n_kv_head=2, n_embd=128, intermediate_size=256)).cuda()
        t = build_model_transform({"_name": "transformer_engine", "replace_norm": fuse, "fuse_swiglu": fuse})
        t.apply(m)
        return m, t

    ids = torch.randint(0, 256, (4, 33), generator=torch.Generator().manual_seed(2)).cuda()
    traces = {}
    for fuse in (True, False):
        m, t = build(fuse)
        assert (t.last_replacements.get("SwiGLU", 0) == 2) == fuse and (t.last_replacements["RMSNorm"] == 5) == fuse
        recipe = amp.FP8Recipe(recipe_type=recipe_name, amax_history_len=4)
        opt = torch.optim.AdamW(m.parameters(), lr=3e-3)
        trace = []
        for _ in range(6):
            opt.zero_grad(set_to_none=True)
            with amp.fp8_autocast(torch.device("cuda"), recipe):
                logits = m(ids[:, :-1])["logits"].float()
                loss = F.cross_entropy(logits.reshape(-1, 256), ids[:, 1:].reshape(-1))
            with amp.fp8_backward(recipe):
                loss.backward()
            opt.step()
            trace.append(loss.item())
        assert all(p.grad is not None for p in m.parameters())
        traces[fuse] = trace
    assert traces[True][-1] < traces[True][0] - 0.3, traces
    assert abs(traces[True][-1] - traces[False][-1]) < 0.15, traces


def test_bias_gradient_comes_out_of_the_amax_pass(amp, monkeypatch):
    from optimus_dl_amd import native
    from optimus_dl_amd.modules.fp8_linear import FP8Linear

    M, K, Nn = 320, 256, 768
    torch.manual_seed(0)
    lin = FP8Linear.from_linear(nn.Linear(K, Nn, bias=True).to("cuda", torch.bfloat16))
    x = seeded_bf16((M, K), 1.0, 1).cuda().requires_grad_(True)
    dy = seeded_bf16((M, Nn), 1e-2, 2)
    recipe = amp.FP8Recipe(recipe_type="tensorwise")
    amax_calls = count_calls(monkeypatch, native, "amax_parts")
    colsum_calls = count_calls(monkeypatch, native, "amax_parts_colsum")
    with recipe.autocast():
        y = lin(x)
    with recipe.backward():
        y.backward(dy.cuda())
    assert colsum_calls == [(M, Nn)] and (M, Nn) not in amax_calls
    want = dy.double().sum(0)
    got = lin.bias.grad.float().cpu().double()
    assert lin.bias.grad.dtype == torch.bfloat16
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-6).all()           # one bf16 rounding of an fp32 sum
    # the codes are those of the plain route: same dx, dw as a bias-free twin fed the same tensors
    twin = FP8Linear.from_linear(nn.Linear(K, Nn, bias=False).to("cuda", torch.bfloat16))
    with torch.no_grad():
        twin.weight.copy_(lin.weight)
    x2 = x.detach().clone().requires_grad_(True)
    with recipe.autocast():
        y2 = twin(x2)
    with recipe.backward():
        y2.backward(dy.cuda())
    assert torch.equal(x.grad, x2.grad) and torch.equal(lin.weight.grad, twin.weight.grad)


@pytest.mark.parametrize("in_dtype", [torch.float32, torch.bfloat16])
def test_fused_layernorm_in_a_gpt2_block(amp, monkeypatch, in_dtype):
    """nn.LayerNorm -> Linear as in a GPT-2 block: the transform re-classes the norm, the Linear takes its maxima,
    outputs and gradients agree with the untouched norm."""
    from optimus_dl_amd import native
    from optimus_dl_amd.modules.model_transforms import build_model_transform

    class Pre(nn.Module):
        def __init__(self):
            super().__init__()
            self.ln = nn.LayerNorm(256)
            self.c_fc = nn.Linear(256, 512)

        def forward(self, x):
            return self.c_fc(self.ln(x))

    torch.manual_seed(0)
    net = Pre().cuda()
    with torch.no_grad():
        net.ln.weight.copy_(torch.linspace(0.5, 1.5, 256))
        net.ln.bias.copy_(torch.linspace(-0.2, 0.2, 256))
    ref = Pre().cuda()
    ref.load_state_dict(net.state_dict())
    t = build_model_transform({"_name": "transformer_engine"})
    t.apply(net)
    assert t.last_replacements["LayerNorm"] == 1 and isinstance(net.ln, nn.LayerNorm)
    build_model_transform({"_name": "transformer_engine", "replace_norm": False}).apply(ref)
    x = (torch.randn(3, 128, 256, generator=torch.Generator().manual_seed(1)) * 2 + 0.3).to(in_dtype).cuda()
    dy = seeded_bf16((3, 128, 512), 1e-2, 2).cuda()
    recipe = amp.FP8Recipe(recipe_type="tensorwise")
    amax_calls = count_calls(monkeypatch, native, "amax_parts")
    outs = {}
    for name, m in (("fused", net), ("plain", ref)):
        xd = x.clone().requires_grad_(True)
        amax_calls.clear()
        with amp.fp8_autocast(torch.device("cuda"), recipe):
            y = m(xd)
        with amp.fp8_backward(recipe):
            y.backward(dy)
        outs[name] = (y.detach(), xd.grad.detach(), m.ln.weight.grad.detach(), m.ln.bias.grad.detach(), m.c_fc.weight.grad.detach())
        assert ((384, 256) in amax_calls) == (name == "plain")          # the normalised activation's own amax pass
    for a, b, tol in zip(outs["fused"], outs["plain"], (1e-2, 2e-2, 2e-2, 2e-2, 1e-2)):
        assert max_rel_err(a, b) <= tol
    assert outs["fused"][1].dtype == in_dtype


def test_gpt2_mlp_with_fused_gelu(amp, monkeypatch):
    """c_proj(gelu(c_fc(x))) with biases: the transform re-classes nn.GELU, c_proj takes the activation's maxima,
    c_fc's backward takes the gradient's, and the results agree with PyTorch's GELU."""
    from optimus_dl_amd import native
    from optimus_dl_amd.modules.model.blocks import GELUMLP
    from optimus_dl_amd.modules.model_transforms import build_model_transform

    def build(fuse):
        torch.manual_seed(0)
        m = GELUMLP(256, 1024, bias=True).to("cuda", torch.bfloat16)
        t = build_model_transform({"_name": "transformer_engine", "fuse_gelu": fuse})
        t.apply(m)
        assert t.last_replacements.get("GELU", 0) == (1 if fuse else 0) and isinstance(m.gelu, nn.GELU)
        return m

    M = 384
    x = seeded_bf16((M, 256), 1.0, 1).cuda()
    dy = seeded_bf16((M, 256), 1e-2, 2).cuda()
    recipe = amp.FP8Recipe(recipe_type="tensorwise")
    amax_calls = count_calls(monkeypatch, native, "amax_parts")
    colsum_calls = count_calls(monkeypatch, native, "amax_parts_colsum")
    fused = step(build(True), recipe, x, dy)
    # x and the two weights by amax_parts; h arrives with its maxima; both grad_outputs go through the amax + column-sum
    # pass because both Linears have a bias (for c_fc it runs for the column sums: the GELU backward left the maxima)
    assert sorted(amax_calls) == sorted([(M, 256), (1024, 256), (256, 1024)]) and colsum_calls == [(M, 256), (M, 1024)]
    amax_calls.clear(); colsum_calls.clear()
    plain = step(build(False), recipe, x, dy)
    assert (M, 1024) in amax_calls and (M, 1024) in colsum_calls
    for a, b in zip(fused, plain):
        assert max_rel_err(a, b) <= 1e-2


# ------------------------------------------------ activation checkpointing around the converted blocks
@pytest.mark.parametrize("fuse", [True, False])
def test_checkpointed_blocks_recompute_the_same_fp8_forward(amp, fuse):
    """The reference wraps blocks in torch.utils.checkpoint (its `activation_checkpoint` transform,
    model_transforms/checkpoint.py:45-81, non-reentrant by default) and runs backward inside the FP8
    backward context: the recomputation then finds the recipe, takes the FP8 path again, saves the same
    tensors, and with per-tensor current scaling reproduces the first forward bit for bit, so every gradient
    equals the one of the run without checkpointing."""
    from torch.utils.checkpoint import checkpoint

    from optimus_dl_amd.modules.model import Llama, LlamaConfig
    from optimus_dl_amd.modules.model_transforms import build_model_transform

    torch.manual_seed(0)
    m = Llama(LlamaConfig(vocab_size=256, n_layer=2, n_head=4, n_kv_head=2, n_embd=128, intermediate_size=256)).cuda()
    build_model_transform({"_name": "fp8_linear", "replace_norm": fuse, "fuse_swiglu": fuse}).apply(m)
    ids = torch.randint(0, 256, (4, 64), generator=torch.Generator().manual_seed(2)).cuda()
    recipe = amp.FP8Recipe(recipe_type="tensorwise")

    def run(ckpt):
        for p in m.parameters():
            p.grad = None
        with amp.fp8_autocast(torch.device("cuda"), recipe):
            x = m.embed(ids)
            for block in m.transformer.h:
                x = checkpoint(block, x, use_reentrant=False) if ckpt else block(x)
            logits = m.lm_head(m.transformer.ln_f(x)).float()
            loss = F.cross_entropy(logits.reshape(-1, 256), ids.reshape(-1))
        with amp.fp8_backward(recipe):
            loss.backward()
        assert recipe.shared_input is None and not recipe.producer_parts        # nothing is kept alive after the step
        return loss.detach(), [p.grad.detach().clone() for p in m.parameters()]

    calls_before = sum(mod.fp8_calls for mod in m.modules() if hasattr(mod, "fp8_calls"))
    loss0, grads0 = run(False)
    calls_plain = sum(mod.fp8_calls for mod in m.modules() if hasattr(mod, "fp8_calls")) - calls_before
    loss1, grads1 = run(True)
    calls_ckpt = sum(mod.fp8_calls for mod in m.modules() if hasattr(mod, "fp8_calls")) - calls_before - calls_plain
    # the Linears inside the blocks ran again on the FP8 path (the recomputation stops at a block's last saved tensor)
    assert calls_plain + 10 <= calls_ckpt <= 2 * calls_plain - 1
    assert torch.equal(loss0, loss1)
    for g0, g1 in zip(grads0, grads1):
        assert torch.equal(g0, g1)


@pytest.mark.parametrize("fuse", [True, False])
def test_a_graph_compiler_steps_around_the_fp8_modules(amp, fuse):
    """The reference can wrap the model in torch.compile (model_transforms/compile.py).  The FP8 modules call the
    native library and are marked so that the tracer leaves them alone: traced with the plain "eager" backend
    (no code generation) the model gives the same bits as without the tracer, forward and backward."""
    import torch._dynamo

    from optimus_dl_amd.modules.model import Llama, LlamaConfig
    from optimus_dl_amd.modules.model_transforms import build_model_transform

    torch.manual_seed(0)
    m = Llama(LlamaConfig(vocab_size=256, n_layer=2, n_head=4, n_kv_head=2, n_embd=128, intermediate_size=256)).cuda()
    build_model_transform({"_name": "fp8_linear", "replace_norm": fuse, "fuse_swiglu": fuse}).apply(m)
    ids = torch.randint(0, 256, (4, 64), generator=torch.Generator().manual_seed(2)).cuda()
    recipe = amp.FP8Recipe(recipe_type="tensorwise")

    def run(model):
        for p in m.parameters():
            p.grad = None
        with amp.fp8_autocast(torch.device("cuda"), recipe):
            logits = model(ids)["logits"].float()
            loss = F.cross_entropy(logits.reshape(-1, 256), ids.reshape(-1))
        with amp.fp8_backward(recipe):
            loss.backward()
        return loss.detach(), [p.grad.detach().clone() for p in m.parameters()]

    before = sum(mod.fp8_calls for mod in m.modules() if hasattr(mod, "fp8_calls"))
    loss0, grads0 = run(m)
    plain_calls = sum(mod.fp8_calls for mod in m.modules() if hasattr(mod, "fp8_calls")) - before
    torch._dynamo.reset()
    compiled = torch.compile(m, backend="eager")
    loss1, grads1 = run(compiled)
    assert sum(mod.fp8_calls for mod in m.modules() if hasattr(mod, "fp8_calls")) - before == 2 * plain_calls
    assert torch.equal(loss0, loss1)
    for g0, g1 in zip(grads0, grads1):
        assert torch.equal(g0, g1)
    torch._dynamo.reset()


@pytest.mark.parametrize("fuse", [True, False])
def test_inference_mode_forward_equals_the_no_grad_forward(amp, fuse):
    """Tensors made under torch.inference_mode keep no version counter, which the hand-over caches key on:
    they must simply miss (every Linear quantises its own input) and the outputs stay the same bits."""
    from optimus_dl_amd.modules.model import Llama, LlamaConfig
    from optimus_dl_amd.modules.model_transforms import build_model_transform

    torch.manual_seed(0)
    m = Llama(LlamaConfig(vocab_size=256, n_layer=2, n_head=4, n_kv_head=2, n_embd=128, intermediate_size=256)).cuda().eval()
    build_model_transform({"_name": "fp8_linear", "replace_norm": fuse, "fuse_swiglu": fuse}).apply(m)
    ids = torch.randint(0, 256, (4, 64), generator=torch.Generator().manual_seed(2)).cuda()
    recipe = amp.FP8Recipe(recipe_type="tensorwise")
    before = sum(mod.fp8_calls for mod in m.modules() if hasattr(mod, "fp8_calls"))
    with torch.no_grad(), amp.fp8_autocast(torch.device("cuda"), recipe):
        want = m(ids)["logits"]
    with torch.inference_mode(), amp.fp8_autocast(torch.device("cuda"), recipe):
        got = m(ids)["logits"]
    assert sum(mod.fp8_calls for mod in m.modules() if hasattr(mod, "fp8_calls")) - before == 2 * 15
    assert torch.equal(got, want)


@pytest.mark.parametrize("tokens,width,hidden", [(32, 128, 256), (160, 192, 384), (1056, 256, 640), (2048, 1024, 4096)])
@pytest.mark.parametrize("kind", ["delayed", "mxfp8", "blockwise"])
def test_whole_mlp_node_changes_no_bit(amp, monkeypatch, kind, tokens, width, hidden):
    """SwiGLU straight to codes against the same MLP as separate nodes, over steps that move the delayed scales: outputs, all
    gradients, histories.  The sizes end inside tiles and K steps; the last one takes wgrad from dY as stored and dX from one GEMM."""
    from optimus_dl_amd.modules import fused
    from optimus_dl_amd.modules.model.blocks import SwiGLUMLP
    from optimus_dl_amd.modules.model_transforms import build_model_transform

    if kind == "blockwise":                       # whole blocks of 128 only
        tokens, width = (tokens + 127) // 128 * 128, (width + 127) // 128 * 128
    nodes = []
    real = fused.swiglu_mlp
    results = {}
    for whole in (True, False):
        monkeypatch.setattr(fused, "swiglu_mlp", (lambda m, x: (nodes.append(1), real(m, x))[1]) if whole else (lambda m, x: None))
        torch.manual_seed(7)
        mlp = build_model_transform({"_name": "fp8_linear"}).apply(SwiGLUMLP(width, hidden).cuda())
        recipe = amp.create_fp8_recipe(kind, "hybrid", amax_history_len=4)
        seen = []
        for step in range(3):
            x = (seeded_bf16((2, tokens // 2, width), 1.0 + step, 3 + step)).cuda().requires_grad_(True)
            mlp.zero_grad()
            with recipe.autocast(), torch.autocast("cuda", dtype=torch.bfloat16):
                y = mlp(x)
            assert (type(y.grad_fn.next_functions[0][0]).__name__ == "_SwiGLUMLPFnBackward") == whole
            with recipe.backward():
                y.backward(seeded_bf16(tuple(y.shape), 1e-3 * (1 + step), 9 + step).cuda())
            seen += [y.detach().clone(), x.grad.clone()] + [p.grad.clone() for p in mlp.parameters()]
        if kind == "delayed":
            seen += [meta.amax_history.clone() for m in (mlp.w1, mlp.w2, mlp.c_proj) for meta in m.fp8_meta.values()]
        results[whole] = seen
    assert nodes and len(results[True]) == len(results[False])
    for a, b in zip(results[True], results[False]):
        assert torch.equal(a, b)


def test_whole_mlp_node_stands_back_for_hooks_and_eval_mode(amp):
    from optimus_dl_amd.modules.fused import swiglu_mlp
    from optimus_dl_amd.modules.model.blocks import SwiGLUMLP
    from optimus_dl_amd.modules.model_transforms import build_model_transform

    mlp = build_model_transform({"_name": "fp8_linear"}).apply(SwiGLUMLP(128, 256).cuda())
    x = seeded_bf16((64, 128), 1.0, 1).cuda().requires_grad_(True)
    seen = []

    def taken(kind="delayed", data=x):
        recipe = amp.create_fp8_recipe(kind, "hybrid", amax_history_len=4)
        with recipe.autocast(), torch.autocast("cuda", dtype=torch.bfloat16):
            return swiglu_mlp(mlp, data) is not None

    assert taken() and taken("mxfp8") and not taken("tensorwise") and not taken("rowwise") and not taken(data=x.detach())
    with torch.no_grad():
        assert not taken()
    hook = mlp.c_proj.register_forward_pre_hook(lambda m, a: seen.append(a[0].shape))
    assert not taken()
    recipe = amp.create_fp8_recipe("delayed", "hybrid", amax_history_len=4)
    with recipe.autocast(), torch.autocast("cuda", dtype=torch.bfloat16):
        mlp(x)
    assert seen == [torch.Size([64, 256])]
    hook.remove()
    handle = torch.nn.modules.module.register_module_forward_hook(lambda m, a, o: None)
    assert not taken()
    handle.remove()
    assert taken()
    mlp.w2.eval()
    assert not taken() and taken("mxfp8")


@pytest.mark.parametrize("rows", [16, 32, 48, 64])
@pytest.mark.parametrize("width,hidden", [(128, 48), (768, 2048), (2048, 5632), (1152, 14336)])
def test_gate_up_and_product_of_a_few_rows_in_one_launch(rows, width, hidden):
    """Bit for bit the two products of the thin kernel (which adds in the same order) and the SwiGLU kernel; from 2048 columns on
    that is the kernel which separate products take by themselves."""
    from optimus_dl_amd import native as N

    x, g, u = seeded_bf16((rows, width), 1.0, rows), seeded_bf16((hidden, width), 0.02, 2), seeded_bf16((hidden, width), 0.02, 3)
    (xq, _, _, _, sx), (gq, _, _, _, sg), (uq, _, _, _, su) = (N.quantize_dynamic(t.cuda(), O.E4M3, 0, True, False) for t in (x, g, u))
    h, parts = N.gemm_swiglu(xq, gq, uq, O.E4M3, O.E4M3, sx, sg, su)
    N.gemm_set_variant(next(i for i, name in enumerate(N.gemm_variants()) if name.startswith("thin")))
    try:
        gate, up = N.gemm_nt(xq, gq, O.E4M3, O.E4M3, sx, sg), N.gemm_nt(xq, uq, O.E4M3, O.E4M3, sx, su)
    finally:
        N.gemm_set_variant(-1)
    assert torch.equal(h, N.swiglu_amax_parts(gate, up)[0])
    assert parts.max().item() == h.float().abs().max().item() and (parts >= 0).all()


@pytest.mark.parametrize("kind", ["tensorwise", "delayed", "rowwise", "mxfp8", "blockwise"])
def test_modules_without_the_cpp_side_of_the_wrappers(amp, monkeypatch, kind):
    """The long way through the wrappers gives the same bits: training step, evaluation and decode step of an MLP."""
    from optimus_dl_amd import native as N

    N.load()
    results = []
    for host in (N._host, N._NoHost()):
        monkeypatch.setattr(N, "_host", host)
        mlp, _ = make_mlp(256, 512)
        recipe = amp.create_fp8_recipe(kind, "hybrid", amax_history_len=4)
        x = seeded_bf16((256, 256), 1.0, 3).cuda().requires_grad_(True)
        with recipe.autocast():
            y = mlp(x)
        with recipe.backward():
            y.backward(seeded_bf16((256, 256), 1e-3, 4).cuda())
        out = [y.detach(), x.grad, *(p.grad for p in mlp.parameters())]
        mlp.eval()
        with recipe.autocast(), torch.no_grad():
            out += [mlp(x), mlp(x[:128]), mlp(x[:32])]
        results.append(out)
    assert all(torch.equal(a, b) for a, b in zip(*results))


def test_decode_step_of_a_swiglu_mlp(amp):
    """Evaluation of a few rows takes the one launch; more rows, hooks and other recipes do not."""
    from optimus_dl_amd.modules import fused

    mlp, _ = make_mlp(256, 512)
    x = seeded_bf16((32, 1, 256), 1.0, 4).cuda()
    recipe = amp.create_fp8_recipe("tensorwise", "hybrid")
    with recipe.autocast(), torch.no_grad():
        h = fused.swiglu_few_rows(mlp, x)
        y = mlp(x)
        many = mlp(x.expand(32, 8, 256).contiguous())
        assert fused.swiglu_few_rows(mlp, x.expand(32, 8, 256)) is None
        assert fused.swiglu_few_rows(mlp, x.expand(32, 2, 256)) is not None
        wide, _ = make_mlp(256, 4352)                         # 64 rows and two rounds of blocks: the separate launches are faster
        assert fused.swiglu_few_rows(wide, x.expand(32, 2, 256)) is None and wide(x.expand(32, 2, 256)).shape == (32, 2, 256)
        assert fused.swiglu_few_rows(wide, x) is not None
        seen = []
        hook = mlp.w2.register_forward_hook(lambda m, a, o: seen.append(o.shape))
        assert fused.swiglu_few_rows(mlp, x) is None
        mlp(x)
        hook.remove()
    assert h.shape == (32, 1, 512) and seen == [torch.Size([32, 1, 512])]
    assert max_rel_err(y.float().cpu(), many[:, :1].float().cpu()) <= 1e-2
    with recipe.autocast():
        assert fused.swiglu_few_rows(mlp, x) is None          # a graph is recorded
    with amp.create_fp8_recipe("rowwise", "hybrid").autocast(), torch.no_grad():
        assert fused.swiglu_few_rows(mlp, x) is None


@pytest.mark.parametrize("whole", [True, False])
def test_delayed_scaling_gives_gate_and_up_weight_gradients_of_their_own(amp, monkeypatch, whole):
    """Every member of a group casts x with its own scale there, so the MLP as one node and the sibling group both multiply twice:
    neither drops a joint product that the other has."""
    from optimus_dl_amd import native
    from optimus_dl_amd.modules import fused
    from optimus_dl_amd.modules.model.blocks import SwiGLUMLP
    from optimus_dl_amd.modules.model_transforms import build_model_transform

    if not whole:
        monkeypatch.setattr(fused, "swiglu_mlp", lambda m, x: None)
    tokens, width, hidden = 560, 1024, 3072
    mlp = build_model_transform({"_name": "fp8_linear"}).apply(SwiGLUMLP(width, hidden).cuda())
    recipe = amp.create_fp8_recipe("delayed", "hybrid", amax_history_len=4)
    x = seeded_bf16((tokens, width), 1.0, 3).cuda().requires_grad_(True)
    with recipe.autocast(), torch.autocast("cuda", dtype=torch.bfloat16):
        y = mlp(x)
    outputs = []
    real = native.gemm_nt
    monkeypatch.setattr(native, "gemm_nt", lambda a, b, *args, **kw: (outputs.append((a.shape[0], b.shape[0])), real(a, b, *args, **kw))[1])
    with recipe.backward():
        y.backward(seeded_bf16((tokens, width), 1e-3, 9).cuda())
    assert outputs.count((hidden, width)) == 2 and (2 * hidden, width) not in outputs


@pytest.mark.parametrize("fmt_x,fmt_w", [(O.E5M2, O.E4M3), (O.E4M3, O.E5M2), (O.E5M2, O.E5M2)])
@pytest.mark.parametrize("rows", [16, 32, 64])
def test_gate_up_and_product_in_every_format(rows, fmt_x, fmt_w):
    """The forms that no recipe asks for, on small multiples of powers of two: every sum of the products is exact."""
    from optimus_dl_amd import native as N

    g = torch.Generator().manual_seed(rows + fmt_x)
    values = torch.tensor([0.0, 0.5, 1.0, -1.0, 2.0, -0.5])
    codes = lambda t, fmt: t.to(O.TORCH_FP8[fmt]).view(torch.uint8).cuda()
    x, gate, up = (values[torch.randint(0, 6, (n, 640), generator=g)] for n in (rows, 52, 52))
    sx, sg, su = (torch.tensor([v]).cuda() for v in (0.125, 0.25, 0.5))
    h, parts = N.gemm_swiglu(codes(x, fmt_x), codes(gate, fmt_w), codes(up, fmt_w), fmt_x, fmt_w, sx, sg, su)
    want = N.swiglu_amax_parts(((x @ gate.t()) * 0.03125).bfloat16().cuda(), ((x @ up.t()) * 0.0625).bfloat16().cuda())[0]
    assert torch.equal(h, want) and parts.max().item() == want.float().abs().max().item()


@pytest.mark.parametrize("rows,hidden,width", [(32, 2048, 768), (64, 3072, 1024), (16, 5632, 1920)])
def test_short_products_of_few_rows_are_as_precise_in_either_order(rows, hidden, width):
    """Below 2048 columns gate and up in one launch add in another order than the separate products (eight partial sums of 128 products
    at a time against one chain of 64 at a time): equally far from 64 bits.  Measured equal to 1e-4; were either sum's own
    rounding to count, eight chains would be off by a third as much as one."""
    from optimus_dl_amd import native as N

    g = torch.Generator(device="cuda").manual_seed(rows)
    a = (torch.randn((rows, width), device="cuda", generator=g) * 20).to(torch.float8_e4m3fn)
    b = (torch.randn((hidden, width), device="cuda", generator=g) * 20).to(torch.float8_e4m3fn)
    exact, one, errors = a.double() @ b.double().t(), torch.ones(1, device="cuda"), []
    for name in ("thin", "128x128x128 4 waves (64x64 per wave)"):
        N.gemm_set_variant(N.gemm_variants().index(next(v for v in N.gemm_variants() if v.startswith(name) and "stages" not in v)))
        try:
            out = N.gemm_nt(a.view(torch.uint8), b.view(torch.uint8), O.E4M3, O.E4M3, one, one, out_dtype=torch.float32)
        finally:
            N.gemm_set_variant(-1)
        errors.append((out.double() - exact).pow(2).mean().sqrt().item())
    assert abs(errors[0] - errors[1]) <= 1e-3 * errors[1]
