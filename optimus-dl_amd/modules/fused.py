"""Producers either side of the FP8 Linear that hand their output's partial maxima to it.

The reference leaves these to PyTorch: ``silu(w1(x)) * w2(x)`` in
optimus_dl/modules/model/blocks/mlp.py:73-76 and RMSNorm in
optimus_dl/modules/model/blocks/layer_norms.py:86-119.  Here one kernel writes the bf16
result and, on the way, the partial maxima of its magnitude; the FP8 Linear that consumes
that very tensor finds them (``FP8Recipe.take_parts``) and casts without an amax pass.
Modules are not replaced but re-classed in place (``module.__class__`` becomes a subclass of
its own class with the forward below), so attributes, parameter names, state-dict keys and
``isinstance`` checks stay what they were.

Without an active FP8 recipe, on the CPU, or for dtypes the kernels do not take, every
forward below is the module's own.
"""

from __future__ import annotations

import torch
import torch.nn as nn
import torch.nn.functional as F

from .. import native
from .amp import state as _state
from .amp.fp8 import FP8Recipe
from .calls import apply, no_graph, untraced
from .fp8_linear import (ROLE_G, ROLE_X, FP8Linear, _converted_input, _Fp8LinearFn, _Fp8LinearGroupFn, _MemberCtx, _product_jobs,
                         _quantise_delayed_for_all, _run_jobs, _wgrad_jobs)


def _bf16_cuda(*tensors: torch.Tensor) -> bool:
    return all(t.is_cuda and t.dtype == torch.bfloat16 for t in tensors)


# ------------------------------------------------------------------------- SwiGLU
class _SwiGLUFn(torch.autograd.Function):
    """h = silu(gate) * up with the roundings of eager bf16 arithmetic; gate and up are kept for
    the backward, h is not (the down projection keeps its FP8 codes only)."""

    @staticmethod
    def forward(ctx, gate: torch.Tensor, up: torch.Tensor, recipe: FP8Recipe):
        h, parts = native.swiglu_amax_parts(gate, up)
        recipe.offer_parts(h, parts)
        ctx.save_for_backward(gate, up)
        ctx.recipe = recipe
        return h

    @staticmethod
    def backward(ctx, dh: torch.Tensor):
        gate, up = ctx.saved_tensors
        if dh.dtype != torch.bfloat16:
            dh = dh.to(torch.bfloat16)
        dgate, dup, parts_g, parts_u = native.swiglu_bwd_amax_parts(dh, gate, up)
        ctx.recipe.offer_parts(dgate, parts_g)
        ctx.recipe.offer_parts(dup, parts_u)
        return dgate, dup, None


@untraced
def swiglu(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    """silu(gate) * up; fused (and feeding the next FP8 Linear) when an FP8 recipe is active."""
    recipe = _state.active_recipe()
    if recipe is None or not _bf16_cuda(gate, up) or gate.shape != up.shape or gate.numel() % 8:
        return F.silu(gate) * up
    return apply(_SwiGLUFn, gate, up, recipe)


# -------------------------------------------------------------- a whole SwiGLU MLP
class _SwiGLUMLPFn(torch.autograd.Function):
    """``c_proj(silu(w1 x) * w2 x)`` as one node, for the recipes that need no amax of the whole tensor before they cast (delayed
    scaling, mxfp8, blockwise).

    The product and its gradients go from the registers of the kernel that computes them straight into codes: h, d_gate and
    d_up are never written in bf16.  Between separate nodes they have to be, since autograd hands tensors over.  Everything
    else is what the three Linears do by themselves (their own forwards and backwards run, on their own saved tensors); gate and
    up never share a weight-gradient GEMM here, nor do they as a sibling group under these recipes (``_joint_wgrad``).

    What one node costs: its saved tensors live until all of it is done, the three weight gradients arrive together, and a
    backward that asks for some of the gradients only (``torch.autograd.grad`` for ``c_proj.weight``, say) computes all of them."""

    @staticmethod
    def forward(ctx, x2d: torch.Tensor, recipe: FP8Recipe, modules: tuple, *weights: torch.Tensor):
        pol = recipe.recipe
        subs, saved = [], []

        def member(x, module, weight, need_x, given=None, jobs=None):
            sub = _MemberCtx((need_x, True, False, False, False, False))
            sub.given_input, sub.y_jobs = given, jobs
            y = _Fp8LinearFn.forward(sub, x, weight, None, module, recipe, torch.bfloat16)
            sub.given_input = sub.y_jobs = None
            sub.span = (len(saved), len(sub.saved_tensors))
            saved.extend(sub.saved_tensors)
            sub.saved_tensors = ()
            subs.append(sub)
            return y

        w1, w2, down = modules
        jobs = _product_jobs(recipe, (w1, w2))
        given = _quantise_delayed_for_all(recipe, x2d, (w1, w2), (True, True))
        gate, up = (member(x2d, w, weight, ctx.needs_input_grad[0], given=g, jobs=jobs)
                    for w, weight, g in ((w1, weights[0], given[0]), (w2, weights[1], given[1])))
        if jobs is not None:
            gate, up = _run_jobs(jobs, pol.fmt_fwd, pol.fmt_fwd, torch.bfloat16, fresh=True)
        if pol.kind == "mxfp8":
            h = native.swiglu_mx_cast(gate, up, pol.fmt_fwd, pol.mx_scale_rule)
        elif pol.kind == "blockwise":
            h = native.swiglu_block_cast(gate, up, pol.fmt_fwd, pol.margin)
        else:
            meta = down._meta(recipe, x2d.device, "fwd")
            meta.note_record(recipe._store)
            h = native.swiglu_cast_delayed(gate, up, meta.scale_of(ROLE_X), pol.fmt_fwd, meta.amax_slot(ROLE_X))
        y = member(gate, down, weights[2], True, given=h)         # (gate: the shape and type of the product)
        ctx.save_for_backward(gate, up, *saved)
        ctx.subs, ctx.recipe = subs, recipe
        return y

    @staticmethod
    def backward(ctx, dy: torch.Tensor):
        gate, up, *tensors = ctx.saved_tensors
        recipe, pol = ctx.recipe, ctx.recipe.recipe
        sub_g, sub_u, sub_d = ctx.subs
        for sub in ctx.subs:
            sub.saved_tensors = tuple(tensors[sub.span[0]:sub.span[0] + sub.span[1]])
        dh, dw_d, *_ = _Fp8LinearFn.backward(sub_d, dy)
        mods = (sub_g.module, sub_u.module)
        if pol.kind == "mxfp8":
            given = native.swiglu_bwd_mx_cast(dh, gate, up, pol.fmt_bwd, pol.mx_scale_rule)
        elif pol.kind == "blockwise":
            given = native.swiglu_bwd_block_cast(dh, gate, up, pol.fmt_bwd, pol.margin)
        elif all(m.training for m in mods):
            metas = [m._meta(recipe, dh.device, "bwd") for m in mods]
            for meta in metas:
                meta.note_record(recipe._store)
            given = native.swiglu_bwd_cast_delayed(dh, gate, up, pol.fmt_bwd, tuple(m.scale_of(ROLE_G) for m in metas),
                                                   tuple(m.amax_slot(ROLE_G) for m in metas), want_transposed=not (sub_g.wgrad_direct and sub_u.wgrad_direct))
        else:                                # put into eval mode since the forward: their histories are left alone
            given = None
        dgate, dup = (gate, up) if given is not None else native.swiglu_bwd_amax_parts(dh, gate, up)[:2]
        pairs, dx_of = _Fp8LinearGroupFn._dgrad_in_one_gemm(ctx, (dgate, dup))
        dx, grads = None, []
        dw_jobs = _wgrad_jobs((sub_g, sub_u), (dgate, dup))
        for i, (sub, g) in enumerate(zip((sub_g, sub_u), (dgate, dup))):
            sub.given_grad = given[i] if given is not None else None
            sub.dx_pairs, sub.dw_jobs = pairs, dw_jobs
            # (block scales: the GEMM that adds into what is there is not the streaming one; a sum of its own is cheaper)
            sub.dx_into = dx if dx is not None and pol.kind == "delayed" else None
            dxi, dw, *_ = _Fp8LinearFn.backward(sub, g)
            sub.given_grad = sub.dx_pairs = sub.dx_into = sub.dw_jobs = None
            if dx is None:
                dx = dxi
            elif dxi is not None and pol.kind != "delayed":
                dx = dx + dxi
            grads.append(dw)
        given = None
        if pairs:
            dx = dx_of(*map(list, zip(*pairs)))
            pairs.clear()                    # the codes of the gradients as stored: their memory is free for the weight gradients
        if dw_jobs:
            grads = _run_jobs(dw_jobs, pol.fmt_bwd, pol.fmt_fwd, sub_g.w_dtype)
        for sub in ctx.subs:
            sub.saved_tensors = ()
        return dx, None, None, *grads, dw_d


_any_global_hook = getattr(torch.nn.modules.module, "_has_any_global_hook", None)


def _runs_as_written(m: FP8Linear) -> bool:
    """Nothing looks at this Linear's input, output or their gradients, and nothing stands in for its forward."""
    return (type(m) is FP8Linear and m.fp8_enabled and m._parameters.get("bias", m) is None and "forward" not in m.__dict__
            and not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks))


@untraced
def swiglu_mlp(mlp: nn.Module, x: torch.Tensor) -> torch.Tensor | None:
    """``mlp(x)`` as one node (``_SwiGLUMLPFn``), or None where its parts have to run on their own: a recipe that
    casts with the amax of the tensor itself, no graph, biases, hooks, a Linear switched off or in eval mode, sizes that
    the kernels do not take, weight gradients that are not FP8 or go straight into ``.grad``."""
    recipe = _state.active_recipe()
    if recipe is None or recipe.recipe.kind not in ("delayed", "mxfp8", "blockwise") or _any_global_hook is None or _any_global_hook():
        return None
    if not torch.is_grad_enabled() or not x.requires_grad or not recipe.wgrad or recipe.fuse_wgrad_accumulation or not recipe.fuse_dgrad_sum:
        return None
    mods = (mlp.w1, mlp.w2, mlp.c_proj)
    w1, w2, down = mods
    if not all(_runs_as_written(m) and m.weight.requires_grad for m in mods):
        return None
    if (torch.get_autocast_dtype("cuda") if torch.is_autocast_enabled("cuda") else x.dtype) != torch.bfloat16:
        return None
    hidden = w1.out_features
    if w2.out_features != hidden or down.in_features != hidden or w1._siblings is None or w1._siblings.misses or w1._siblings is not w2._siblings:
        return None
    if not (w1._fp8_eligible(x) and w2._fp8_eligible(x)) or not down.weight.is_cuda or down.weight.dtype not in (torch.bfloat16, torch.float32):
        return None
    delayed = recipe.recipe.kind == "delayed"
    out_mult = {"delayed": 16, "mxfp8": 32, "blockwise": 128}[recipe.recipe.kind]
    if hidden % (16 if delayed else 128) or down.out_features % out_mult or (delayed and not all(m.training for m in mods)):
        return None
    x2d = x.reshape(-1, w1.in_features)
    if x2d.dtype != torch.bfloat16 or not x2d.is_contiguous():
        x2d = _converted_input(recipe, x2d, torch.bfloat16)
    for m in mods:
        m.__dict__["fp8_calls"] += 1
        m._note_grad_mode()
    y = apply(_SwiGLUMLPFn, x2d, recipe, mods, w1.weight, w2.weight, down.weight)
    return y.reshape(*x.shape[:-1], down.out_features)


@untraced
def swiglu_few_rows(mlp: nn.Module, x: torch.Tensor) -> torch.Tensor | None:
    """``silu(w1 x) * w2 x`` of a decode step in one launch (``native.gemm_swiglu``), or None: only per-tensor current scaling,
    no graph, few rows (``native.gemm_swiglu_pays``), no biases, no hooks.  The value of the separate modules; to the last bit where
    their products take the thin kernel (``native.gemm_swiglu``)."""
    recipe = _state.active_recipe()
    if recipe is None or recipe.recipe.kind != "tensorwise" or not no_graph() or _any_global_hook is None or _any_global_hook():
        return None
    w1, w2 = mlp.w1, mlp.w2
    if not (_runs_as_written(w1) and _runs_as_written(w2)):       # (whatever may have been put in their place, a wrapper say)
        return None
    k = w1.in_features
    if w2.out_features != w1.out_features or w2.in_features != k or not native.gemm_swiglu_pays(x.numel() // max(k, 1), w1.out_features, k):
        return None
    if (torch.get_autocast_dtype("cuda") if torch.is_autocast_enabled("cuda") else x.dtype) != torch.bfloat16:
        return None
    w2_weight = w2.weight
    if not w1._fp8_eligible(x) or not w2_weight.is_cuda or w2_weight.dtype not in (torch.bfloat16, torch.float32):
        return None
    x2d = x.reshape(-1, k)
    if x2d.dtype != torch.bfloat16 or not x2d.is_contiguous():
        x2d = _converted_input(recipe, x2d, torch.bfloat16)
    pol = recipe.recipe
    parts = recipe.take_parts(x2d)
    xq, _, _, _, sx_inv = (native.quantise_small(x2d, pol.fmt_fwd, pol.margin) if parts is None
                           else native.cast_dynamic(x2d, parts, pol.fmt_fwd, pol.margin, want_transposed=False))
    codes = []
    for m, weight in ((w1, w1.weight), (w2, w2_weight)):
        m.__dict__["fp8_calls"] += 1
        m._note_grad_mode()
        codes.append(m._tensor_weight(weight, recipe, need_t=recipe.cache_weights and x2d.requires_grad))
    (g, _, sg_inv), (u, _, su_inv) = codes
    h, parts = native.gemm_swiglu(xq, g, u, pol.fmt_fwd, pol.fmt_fwd, sx_inv, sg_inv, su_inv)
    h = h.reshape(*x.shape[:-1], w1.out_features)
    recipe.offer_parts(h, parts)
    return h


# ---------------------------------------------------------------- in-place re-classing
# A module is fused by giving it a subclass of its own class with the fused forward mixed in: same object, same
# parameters, same state-dict keys, isinstance() checks keep working.  The subclass is made on the fly, so pickling
# it by name would find the original class instead: the mixins carry a __reduce_ex__ that rebuilds the subclass
# from (original class, mixin) -- copy.deepcopy (EMA copies of a model) and torch.save of a whole module both work.
_RECLASSED: dict[tuple[type, type], type] = {}


def _fused_class(base: type, mixin: type) -> type:
    key = (base, mixin)
    cls = _RECLASSED.get(key)
    if cls is None:
        cls = type(base.__name__, (mixin, base), {"__module__": base.__module__})
        _RECLASSED[key] = cls
    return cls


def _rebuild_fused(base: type, mixin: type):
    cls = _fused_class(base, mixin)
    return cls.__new__(cls)


class _Reclassed:
    def __reduce_ex__(self, protocol):
        mro = type(self).__mro__                      # (made-up subclass, mixin, _Reclassed, original class, ...)
        return _rebuild_fused, (mro[mro.index(_Reclassed) + 1], mro[1]), self.__dict__


class _FusedSwiGLUForward(_Reclassed):
    """Mixed into the class of an MLP with ``w1`` (gate), ``w2`` (up) and ``c_proj`` (down)."""

    _odl_fused_swiglu = True

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if _state.active_recipe() is None or not x.is_cuda:
            return super().forward(x)
        if torch.is_grad_enabled():
            y = swiglu_mlp(self, x)
            if y is not None:
                return y
            h = None
        else:
            h = swiglu_few_rows(self, x)
        return self.c_proj(swiglu(self.w1(x), self.w2(x)) if h is None else h)


def fuse_swiglu_mlp(mlp: nn.Module) -> bool:
    """Re-class ``mlp`` in place so that its forward is the fused one.  Only modules whose three
    projections are FP8 Linears named as in the reference's SwiGLUMLP (mlp.py:47-49) qualify."""
    if getattr(mlp, "_odl_fused_swiglu", False):
        return False
    if not all(isinstance(getattr(mlp, n, None), FP8Linear) for n in ("w1", "w2", "c_proj")):
        return False
    cls = mlp.__class__
    mlp.__class__ = _fused_class(cls, _FusedSwiGLUForward)
    return True


# ------------------------------------------------------------------------ RMSNorm
class _RMSNormFn(torch.autograd.Function):
    """y = (x * rsqrt(mean(x^2) + eps)) * weight rounded once to bf16."""

    @staticmethod
    def forward(ctx, x: torch.Tensor, weight: torch.Tensor, eps: float, recipe: FP8Recipe):
        y, rstd, parts = native.rmsnorm_amax_parts(x, weight, eps)
        recipe.offer_parts(y, parts)
        ctx.save_for_backward(x, weight, rstd)
        return y

    @staticmethod
    def backward(ctx, dy: torch.Tensor):
        x, weight, rstd = ctx.saved_tensors
        if dy.dtype != torch.bfloat16:
            dy = dy.to(torch.bfloat16)
        dx, dw = native.rmsnorm_bwd(dy, x, weight, rstd)
        return (dx if ctx.needs_input_grad[0] else None), (dw.to(weight.dtype) if ctx.needs_input_grad[1] else None), None, None


@untraced
def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor | None:
    """Fused RMSNorm when an FP8 recipe is active and the kernel takes the input; else None."""
    recipe = _state.active_recipe()
    if recipe is None or not x.is_cuda or x.dtype not in (torch.bfloat16, torch.float32):
        return None
    if x.dtype != torch.bfloat16 and not (torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") == torch.bfloat16):
        return None                    # an fp32 result is expected downstream: the module's own forward
    cols = x.shape[-1]
    if cols % 8 or cols < 8 or cols > 8192 or weight.numel() != cols or x.numel() == 0:
        return None
    return apply(_RMSNormFn, x, weight, float(eps), recipe)


class _FusedRMSNormForward(_Reclassed):
    """Mixed into the class of an RMSNorm with ``weight`` and ``eps`` (layer_norms.py:64-67).

    Under an FP8 recipe the output is bf16 whatever the input dtype: the recipe's context nests
    a bf16 autocast (fp8.py:488-493), so the Linear that follows would round an fp32 output to
    bf16 anyway; the values are the same, the fp32 copy is never written."""

    _odl_fused_rmsnorm = True

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        y = rmsnorm(x, self.weight, self.eps)
        return super().forward(x) if y is None else y


def fuse_rmsnorm(norm: nn.Module) -> bool:
    if getattr(norm, "_odl_fused_rmsnorm", False):
        return False
    w = getattr(norm, "weight", None)
    if not isinstance(w, torch.Tensor) or w.dim() != 1 or not hasattr(norm, "eps"):
        return False
    cls = norm.__class__
    norm.__class__ = _fused_class(cls, _FusedRMSNormForward)
    return True


# ---------------------------------------------------------------------- LayerNorm
class _LayerNormFn(torch.autograd.Function):
    """y = layer_norm(x) * weight + bias rounded once to bf16."""

    @staticmethod
    def forward(ctx, x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None, eps: float, recipe: FP8Recipe):
        y, mean, rstd, parts = native.layernorm_amax_parts(x, weight, bias, eps)
        recipe.offer_parts(y, parts)
        ctx.save_for_backward(x, weight, mean, rstd)
        ctx.bias_dtype = None if bias is None else bias.dtype
        return y

    @staticmethod
    def backward(ctx, dy: torch.Tensor):
        x, weight, mean, rstd = ctx.saved_tensors
        if dy.dtype != torch.bfloat16:
            dy = dy.to(torch.bfloat16)
        dx, dw, db = native.layernorm_bwd(dy, x, weight, mean, rstd)
        return (dx if ctx.needs_input_grad[0] else None, dw.to(weight.dtype) if ctx.needs_input_grad[1] else None,
                db.to(ctx.bias_dtype) if ctx.bias_dtype is not None and ctx.needs_input_grad[2] else None, None, None)


@untraced
def layernorm(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None, eps: float) -> torch.Tensor | None:
    """Fused LayerNorm when an FP8 recipe is active and the kernel takes the input; else None."""
    recipe = _state.active_recipe()
    if recipe is None or not x.is_cuda or x.dtype not in (torch.bfloat16, torch.float32):
        return None
    if x.dtype != torch.bfloat16 and not (torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") == torch.bfloat16):
        return None
    cols = x.shape[-1]
    if cols % 8 or cols < 8 or cols > 4096 or weight is None or weight.numel() != cols or x.numel() == 0:
        return None
    return apply(_LayerNormFn, x, weight, bias, float(eps), recipe)


class _FusedLayerNormForward(_Reclassed):
    """Mixed into the class of a LayerNorm over the last axis: ``torch.nn.LayerNorm`` (``normalized_shape``
    of one dimension, affine) or the reference's bias-optional one (layer_norms.py:21-47, eps 1e-5).
    Output dtype under an FP8 recipe: as for the fused RMSNorm."""

    _odl_fused_layernorm = True

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        y = layernorm(x, self.weight, getattr(self, "bias", None), getattr(self, "eps", 1e-5))
        return super().forward(x) if y is None else y


def fuse_layernorm(norm: nn.Module) -> bool:
    if getattr(norm, "_odl_fused_layernorm", False):
        return False
    w = getattr(norm, "weight", None)
    if not isinstance(w, torch.Tensor) or w.dim() != 1:
        return False                       # no affine weight, or normalisation over several axes
    shape = getattr(norm, "normalized_shape", None)
    if shape is not None and tuple(shape) != (w.numel(),):
        return False
    cls = norm.__class__
    norm.__class__ = _fused_class(cls, _FusedLayerNormForward)
    return True


# --------------------------------------------------------------------------- GELU
class _GeluFn(torch.autograd.Function):
    """Exact (erf) GELU of a bf16 tensor, its input kept for the backward."""

    @staticmethod
    def forward(ctx, x: torch.Tensor, recipe: FP8Recipe, sums: bool):
        y, parts = native.gelu_amax_parts(x)
        recipe.offer_parts(y, parts)
        ctx.save_for_backward(x)
        ctx.recipe, ctx.sums = recipe, sums
        return y

    @staticmethod
    def backward(ctx, dy: torch.Tensor):
        (x,) = ctx.saved_tensors
        if dy.dtype != torch.bfloat16:
            dy = dy.to(torch.bfloat16)
        if ctx.sums:
            dx, parts, slabs = native.gelu_bwd_slabs(dy, x)
        else:
            (dx, parts), slabs = native.gelu_bwd_amax_parts(dy, x), None
        ctx.recipe.offer_parts(dx, parts, slabs)
        return dx, None, None


# what ``_forward_fp8`` may put between a Linear's product and what its caller gets
_VIEW_NODES = frozenset(("ViewBackward0", "UnsafeViewBackward0", "ReshapeAliasBackward0", "AliasBackward0"))


def _gradient_is_summed(x: torch.Tensor, recipe: FP8Recipe) -> bool:
    """Whether the gradient of x goes to an FP8 Linear with a bias, under a recipe that takes sums of its columns from the kernel that makes
    it.  Sums cost that kernel up to a tenth of its time (16384 x 3072: 55.0 us, 60.4 with them) and spare such a Linear a pass over dx; they
    would be made for nobody in front of a Linear without a bias, one that stays in bf16, or anything else.  Forward and backward of the
    MLP on 16384 tokens, without sums / with them where they are used, us: 2048 -> 8192 (dW reads dY as stored) 1715 / 1681, 768 -> 3072
    528 / 495; without a bias 1640 / 1640."""
    node = x.grad_fn
    if node is None or recipe.recipe.kind != "tensorwise":
        return False
    if type(node).__name__ in _VIEW_NODES:
        node = node.next_functions[0][0]
    return isinstance(getattr(node, "module", None), FP8Linear) and getattr(node, "has_bias", False) and getattr(node, "recipe", None) is recipe


@untraced
def gelu(x: torch.Tensor) -> torch.Tensor | None:
    """Fused GELU when an FP8 recipe is active and the input is a bf16 GPU tensor; else None."""
    recipe = _state.active_recipe()
    if recipe is None or not _bf16_cuda(x) or x.numel() % 8 or x.numel() == 0:
        return None
    return apply(_GeluFn, x, recipe, _gradient_is_summed(x, recipe))


class _FusedGeluForward(_Reclassed):
    """Mixed into the class of an ``nn.GELU`` with the exact (erf) form, the activation of the
    reference's GELUMLP (mlp.py:141-157)."""

    _odl_fused_gelu = True

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        y = gelu(x)
        return super().forward(x) if y is None else y


def fuse_gelu(act: nn.Module) -> bool:
    if getattr(act, "_odl_fused_gelu", False) or not isinstance(act, nn.GELU) or getattr(act, "approximate", "none") != "none":
        return False
    cls = act.__class__
    act.__class__ = _fused_class(cls, _FusedGeluForward)
    return True
