"""
``Float8Linear`` and the model swap.

The module keeps the ``nn.Linear`` surface (same ``weight`` / ``bias`` Parameters, same state-dict keys) and
routes its matmuls through one ``torch.autograd.Function`` that quantises the operands with the HIP cast
kernels and multiplies them on the fp8 matrix cores.  This is the native counterpart of what the reference
obtains from ``torchao.float8.convert_to_float8_training`` (reference call site:
src/olmo_core/float8/__init__.py:133-150).

Per linear and training step (M tokens, weight [N, K]):

    output      y  [M, N] = q(x)  [M, K] . q(W)  [N, K]^T
    grad_input  gx [M, K] = q(go) [M, N] . q(W)^T [K, N]^T
    grad_weight gW [N, K] = q(go)^T [N, M] . q(x)^T [K, M]^T

Every GEMM reads both operands K-contiguous, so the casts emit row-major and/or transposed fp8 copies:
tensorwise casts emit both orientations from one pass with one scale; axiswise ("rowwise" recipes) casts
emit a per-row-scaled row-major copy for operands reduced along their rows and a per-column-scaled
transposed copy for operands reduced along their columns.
"""

from __future__ import annotations

from typing import Callable, Optional, Tuple

import torch
import torch.nn as nn

from . import ops, plan
from .native_config import CastConfig, Float8LinearConfig, ScalingGranularity, ScalingType

__all__ = ["Float8Linear", "convert_to_float8_training", "float8_linear_function", "float8_projections"]


def needs_autograd(*tensors: torch.Tensor) -> bool:
    """Whether a call on these tensors has to go through an autograd function: some gradient is wanted, or
    forward-mode differentiation or a transform (vmap, torch.func.grad, ...) is on, which the function refuses by name
    where plain kernels would drop the tangent or stumble over a tensor without storage."""
    if torch.is_grad_enabled() and any(t.requires_grad for t in tensors):
        return True
    return torch.autograd.forward_ad._current_level >= 0 or torch._C._are_functorch_transforms_active()


def _is_tensorwise(c: CastConfig) -> bool:
    return c.scaling_type is ScalingType.DYNAMIC and c.scaling_granularity is ScalingGranularity.TENSORWISE


def _is_axiswise(c: CastConfig) -> bool:
    return c.scaling_type is ScalingType.DYNAMIC and c.scaling_granularity is ScalingGranularity.AXISWISE


def _is_disabled(c: CastConfig) -> bool:
    return c.scaling_type is ScalingType.DISABLED


def _shared_tensorwise(a: CastConfig, b: CastConfig) -> bool:
    """Two uses of one tensor that quantise identically (one scale, one dtype): cast once, emit both layouts."""
    return _is_tensorwise(a) and _is_tensorwise(b) and a.target_dtype == b.target_dtype


def _shared_axiswise(a: CastConfig, b: CastConfig) -> bool:
    """Two uses of one tensor, one scaled per row and one per column, in the same fp8 type: both copies come out
    of one two-product cast."""
    return _is_axiswise(a) and _is_axiswise(b) and a.target_dtype == b.target_dtype


def _rows_operand(x: torch.Tensor, c: CastConfig, pow2: bool) -> Tuple[torch.Tensor, torch.Tensor]:
    """Operand reduced along its rows' elements (K = last dim of x): row-major fp8 + scale [1] or [rows]."""
    if _is_tensorwise(c):
        q, _, s = ops.cast_tensorwise(x, c.target_dtype, pow2=pow2, want_rowmajor=True, want_transposed=False)
        return q, s
    return ops.cast_rowwise(x, c.target_dtype, pow2=pow2)


def _cols_operand(x: torch.Tensor, c: CastConfig, pow2: bool) -> Tuple[torch.Tensor, torch.Tensor]:
    """Operand whose K is x's first dim: transposed fp8 [cols, rows padded with zeros] + scale [1] or [cols]."""
    if _is_tensorwise(c):
        _, q_t, s = ops.cast_tensorwise(x, c.target_dtype, pow2=pow2, want_rowmajor=False, want_transposed=True,
                                       whole_steps=True)
        return q_t, s
    return ops.cast_colwise_t(x, c.target_dtype, pow2=pow2)


def _saves_quantised(c: Float8LinearConfig, need_gx: bool, need_gw: bool) -> Tuple[bool, bool]:
    """Whether the forward keeps the transposed fp8 copy (+ scale) of x / of the weight for the backward instead
    of the high-precision tensor: possible when forward and backward quantise that tensor identically."""
    if _is_disabled(c.cast_config_input):
        return False, False
    ci, ciw = c.cast_config_input, c.cast_config_input_for_grad_weight
    cw, cwi = c.cast_config_weight, c.cast_config_weight_for_grad_input
    x_is_q = need_gw and (_shared_tensorwise(ci, ciw) or _shared_axiswise(ci, ciw))
    w_is_q = need_gx and (_shared_tensorwise(cw, cwi) or _shared_axiswise(cw, cwi))
    return x_is_q, w_is_q


def _input_operands(x2, c: Float8LinearConfig, pow2: bool, share_x: bool):
    """``(xq, sx, x_saved)`` for the forward GEMM: the by-rows operand, its scale, and what the backward keeps."""
    ci = c.cast_config_input
    x_saved = None
    if _is_tensorwise(ci):
        xq, xq_t, sx = ops.cast_tensorwise(x2, ci.target_dtype, pow2=pow2, want_rowmajor=True, want_transposed=share_x,
                                           whole_steps=True)
        if share_x:
            x_saved = (xq_t, sx)
    elif share_x:  # per-row copy for this GEMM, per-column transposed copy for grad_weight, one cast
        xq, sx, xq_t, sxc = ops.cast_rows_and_colwise_t(x2, ci.target_dtype, pow2=pow2)
        x_saved = (xq_t, sxc)
    else:
        xq, sx = ops.cast_rowwise(x2, ci.target_dtype, pow2=pow2)
    return xq, sx, x_saved


def _weight_operands(weight, c: Float8LinearConfig, pow2: bool, share_w: bool, rows: int, weight_scale=None, weight_ops=None):
    """``(wq, sw, w_saved)`` for the forward GEMM of ``rows`` rows: the weight's by-rows operand, its scale(s), and what the backward
    keeps for grad_input (``(q_t, scale)`` or ``None``: keep the weight itself)."""
    w_saved = None
    if weight_ops is not None:
        wq, wq_t, sw = weight_ops
        if share_w:
            w_saved = (wq_t, sw)
    elif _is_tensorwise(c.cast_config_weight):
        wq, wq_t, sw = ops.cast_tensorwise(
            weight, c.cast_config_weight.target_dtype, pow2=pow2, want_rowmajor=True, want_transposed=share_w,
            scale=weight_scale,
        )
        if share_w:
            w_saved = (wq_t, sw)
    elif share_w:
        wq, sw, wq_t, swc = ops.cast_rows_and_colwise_t(weight, c.cast_config_weight.target_dtype, pow2=pow2)
        w_saved = (wq_t, swc)
    else:
        wq, sw = ops.cast_rowwise(weight, c.cast_config_weight.target_dtype, pow2=pow2, product_rows=rows)
    return wq, sw, w_saved


def _forward_operands(x2, weights, c: Float8LinearConfig, scales, w_ops, share_x: bool, share_w: bool):
    """:func:`_input_operands` of ``x2`` and :func:`_weight_operands` of every weight: ``(xq, sx, x_saved, [(wq, sw,
    w_saved), ...])``.  Tensors that are cast alike share their launches."""
    pow2 = c.round_scales_to_power_of_2
    ci, cw = c.cast_config_input, c.cast_config_weight
    if ci.target_dtype == cw.target_dtype and any(o is None for o in w_ops):
        if _is_tensorwise(ci) and _is_tensorwise(cw):
            more = [(w, dict(want_transposed=share_w, scale=s)) for w, s, o in zip(weights, scales, w_ops) if o is None]
            (xq, xq_t, sx), *made = ops.cast_tensorwise(x2, ci.target_dtype, pow2=pow2, want_transposed=share_x, whole_steps=True,
                                                        more=more)
            made = iter(made)
            ws = [next(made) if o is None else o for o in w_ops]
            return xq, sx, (xq_t, sx) if share_x else None, [(q, s, (q_t, s) if share_w else None) for q, q_t, s in ws]
        if _is_axiswise(ci) and _is_axiswise(cw) and share_x and share_w and all(o is None for o in w_ops):
            (xq, sx, xq_t, sxc), *made = ops.cast_rows_and_colwise_t(x2, ci.target_dtype, pow2=pow2, more=weights)
            return xq, sx, (xq_t, sxc), [(q, s, (q_t, sc)) for q, s, q_t, sc in made]
    return (*_input_operands(x2, c, pow2, share_x),
            [_weight_operands(w, c, pow2, share_w, x2.shape[0], s, o) for w, s, o in zip(weights, scales, w_ops)])


def _forward_impl(x2, weight, c: Float8LinearConfig, weight_scale, need_gx: bool, need_gw: bool, weight_ops=None):
    """y = x2 @ weight^T in float8.  Returns ``(y, x_saved, w_saved)``: the tensors the backward needs for x and
    for the weight, each either ``(q_t, scale)`` (see :func:`_saves_quantised`) or ``None`` (keep the input).
    ``weight_ops``: ``(q, q_t, scale)`` of the weight kept by the module (:meth:`Float8Linear.weight_operands`);
    the weight is then not quantised here."""
    if _is_disabled(c.cast_config_input):
        return torch.mm(x2, weight.t().to(x2.dtype)), None, None
    share_x, share_w = _saves_quantised(c, need_gx, need_gw)
    xq, sx, x_saved, ((wq, sw, w_saved),) = _forward_operands(x2, (weight,), c, (weight_scale,), (weight_ops,), share_x, share_w)
    return ops.gemm_fp8(xq, sx, wq, sw, out_dtype=x2.dtype), x_saved, w_saved


def _grad_operands(gos, c: Float8LinearConfig, need_gx: bool, need_gws):
    """Each grad_output's operands ``(rows, cols)`` for the grad_input and the grad_weight GEMM where both are wanted and
    quantise it alike (all of them share their launches), else ``(None, None)``."""
    pow2 = c.round_scales_to_power_of_2
    cg, cgw = c.cast_config_grad_output, c.cast_config_grad_output_for_grad_weight
    made = [(None, None)] * len(gos)
    todo = [i for i, (go, need) in enumerate(zip(gos, need_gws)) if go is not None and need_gx and need]
    if todo and _shared_tensorwise(cg, cgw):
        kw = dict(want_transposed=True, whole_steps=True)
        for i, (q, q_t, s) in zip(todo, ops.cast_tensorwise_batch([(gos[i], kw) for i in todo], cg.target_dtype, pow2=pow2)):
            made[i] = (q, s), (q_t, s)
    elif todo and _shared_axiswise(cg, cgw):
        for i, (q, rs, q_t, cs) in zip(todo, ops.cast_rows_and_colwise_t_batch([gos[i] for i in todo], cg.target_dtype, pow2=pow2)):
            made[i] = (q, rs), (q_t, cs)
    return made


def _backward_impl(go2, c: Float8LinearConfig, N: int, x_dtype, w_dtype, x_part, w_part, x_is_q: bool, w_is_q: bool,
                   need_gx: bool, need_gw: bool, gx_into=None, go_operands=None):
    """grad_input and grad_weight from grad_output ``go2 [M, N]``; ``x_part`` / ``w_part`` are what the forward
    kept: ``(q_t, scale)`` if the flag says so, else ``(tensor,)``.  ``gx_into``: a ``[M, K]`` tensor of ``x_dtype``
    that this linear's grad_input is added to (the bits of ``gx_into + grad_input``, formed in the GEMM's epilogue)
    and that is returned as ``gx``.  ``go_operands``: what :func:`_grad_operands` made of ``go2``."""
    pow2 = c.round_scales_to_power_of_2
    if go2.dtype != x_dtype:
        go2 = go2.to(x_dtype)
    cg, cgw = c.cast_config_grad_output, c.cast_config_grad_output_for_grad_weight
    # grad_output is quantised once if both backward GEMMs want the same cast
    go_rows, go_cols = go_operands if go_operands is not None else _grad_operands([go2], c, need_gx, [need_gw])[0]

    gx = gw = None
    products = []
    if need_gx:
        if _is_disabled(cg):
            gx = torch.mm(go2, w_part[0].to(go2.dtype))
            if gx_into is not None:
                gx = gx_into.add_(gx)
        else:
            args = _grad_input_product(go2, c, N, go_rows, w_part, w_is_q)
            if gx_into is None:
                products.append(args)
            else:
                gx = ops.gemm_fp8(*args[:4], k=N, out_dtype=x_dtype, out=gx_into, accumulate=True)
    if need_gw:
        if _is_disabled(cgw):
            gw = torch.mm(go2.t(), x_part[0].to(go2.dtype))
        else:
            products.append(_grad_weight_product(go2, c, go_cols, x_part, x_is_q, w_dtype))
    if products:
        made = ops.gemm_fp8_products(products, out_dtype=x_dtype)
        if need_gw and not _is_disabled(cgw):
            gw = made.pop()
        if made:
            gx = made.pop()
    if gw is not None and gw.dtype != w_dtype:
        gw = gw.to(w_dtype)
    return gx, gw


def _grad_input_product(go2, c: Float8LinearConfig, N: int, go_rows, w_part, w_is_q: bool, add: bool = False):
    """The grad_input term of one linear as :func:`ops.gemm_fp8_batch` takes it."""
    pow2 = c.round_scales_to_power_of_2
    if go_rows is None:
        go_rows = _rows_operand(go2, c.cast_config_grad_output, pow2)
    w_op = w_part if w_is_q else _cols_operand(w_part[0], c.cast_config_weight_for_grad_input, pow2)
    return (go_rows[0], go_rows[1], w_op[0], w_op[1], N, add)


def _grad_weight_product(go2, c: Float8LinearConfig, go_cols, x_part, x_is_q: bool, w_dtype):
    """The grad_weight of one linear as :func:`ops.gemm_fp8_batch` takes it (written as float32 for a float32 weight)."""
    pow2 = c.round_scales_to_power_of_2
    if go_cols is None:
        go_cols = _cols_operand(go2, c.cast_config_grad_output_for_grad_weight, pow2)
    x_op = x_part if x_is_q else _cols_operand(x_part[0], c.cast_config_input_for_grad_weight, pow2)
    return (go_cols[0], go_cols[1], x_op[0], x_op[1], None, False, w_dtype)


def _options(c: Float8LinearConfig) -> tuple:
    """What of a config the launches of a linear follow from."""
    out = [c.round_scales_to_power_of_2]
    for cc in (c.cast_config_input, c.cast_config_input_for_grad_weight, c.cast_config_weight, c.cast_config_weight_for_grad_input,
               c.cast_config_grad_output, c.cast_config_grad_output_for_grad_weight):
        out += (id(cc.scaling_type), id(cc.scaling_granularity), cc.target_dtype)  # (ids of members of enumerations)
    return tuple(out)


def _planned_forward(x2, weights, c: Float8LinearConfig, scales, w_ops, need_gx: bool, need_gw: bool):
    """:func:`_shared_input_forward` from a plan: ``(ys, kept, plan)`` or ``None``.  Only where all that the backward takes is
    quantised here."""
    if need_gx and any(o is not None for o in w_ops):
        return None
    n = len(weights)

    def recorded(px, *rest):
        given = [rest[2 * n + 3 * i:2 * n + 3 * i + 3] for i in range(n)]
        ys, x_saved, w_saved = _shared_input_forward(px, rest[:n], c, rest[n:2 * n], [g if g[0] is not None else None for g in given],
                                                     need_gx, need_gw)
        if (need_gw and x_saved is None) or (need_gx and None in w_saved):
            raise plan.Unplannable("an input is kept")
        return ys, (x_saved if need_gw else None, w_saved if need_gx else None)

    inputs = [x2, *weights, *scales]
    for o in w_ops:
        inputs += (None, None, None) if o is None else o
    return plan.call(recorded, inputs, ("linears", n, need_gx, need_gw, _options(c)), own=3 * n)


def _planned_backward(ctx, gos, ns, need_gx: bool, need_gws):
    """``(gx, gws)`` of a forward that ran from a plan (grad_weights in the type of x; ``None`` where nothing is wanted)."""
    c, M, (kept,) = ctx.config, ctx.M, ctx.saved_tensors
    gos = [None if go is None else go.reshape(M, N) for go, N in zip(gos, ns)]
    gos = [go if go is None or (go.dtype == ctx.x_dtype and go.is_contiguous()) else go.to(ctx.x_dtype).contiguous() for go in gos]
    order = [i for i in reversed(range(len(gos))) if gos[i] is not None]
    wanted = [i for i in order if need_gws[i]]
    if not order:
        return None, [None] * len(gos)

    def products(gos_, saved):
        x_part, w_parts = saved
        made = _grad_operands(gos_, c, need_gx, need_gws)
        ps = [_grad_input_product(gos_[i], c, ns[i], made[i][0], w_parts[i], True, add=i != order[0]) for i in order if need_gx]
        ps += [_grad_weight_product(gos_[i], c, made[i][1], x_part, True, ctx.w_dtypes[i]) for i in wanted]
        return ops.gemm_fp8_products(ps, out_dtype=ctx.x_dtype)

    def recorded(slab, *places):
        return products(places, ctx.plan.saved_places(slab)), None

    done = plan.call(recorded, [kept, *gos], ("backward", need_gx, tuple(need_gws)), within=ctx.plan)
    outs = done[0] if done is not None else products(gos, ctx.plan.saved_tensors(kept))
    outs = list(outs)
    gx = outs.pop(0) if need_gx else None
    gws = [None] * len(gos)
    for i, gw in zip(wanted, outs):
        gws[i] = gw
    return gx, gws


def _fp8_backward(c: Float8LinearConfig) -> bool:
    return not (_is_disabled(c.cast_config_input) or _is_disabled(c.cast_config_grad_output)
                or _is_disabled(c.cast_config_grad_output_for_grad_weight))


class _Float8Matmul(torch.autograd.Function):
    """y = x @ W^T with float8 operands; x [M, K] and W [N, K] in high precision."""

    @staticmethod
    def forward(ctx, x2: torch.Tensor, weight: torch.Tensor, config: Float8LinearConfig, weight_scale=None,
                weight_ops=None):
        need_gx, need_gw = ctx.needs_input_grad[0], ctx.needs_input_grad[1]
        done = _planned_forward(x2, (weight,), config, (weight_scale,), (weight_ops,), need_gx, need_gw) if _fp8_backward(config) else None
        ctx.plan = None
        if done is not None:
            (y,), kept, ctx.plan = done
            ctx.config, ctx.M, ctx.N, ctx.x_dtype, ctx.w_dtype = config, x2.shape[0], weight.shape[0], x2.dtype, weight.dtype
            ctx.w_dtypes = [weight.dtype]
            ctx.save_for_backward(kept)
            return y
        y, x_saved, w_saved = _forward_impl(x2, weight, config, weight_scale, need_gx, need_gw, weight_ops)
        ctx.config = config
        ctx.x_dtype, ctx.w_dtype = x2.dtype, weight.dtype
        ctx.shapes = (x2.shape[0], x2.shape[1], weight.shape[0])
        ctx.x_is_q, ctx.w_is_q = x_saved is not None, w_saved is not None
        to_save = []
        if need_gw:
            to_save += list(x_saved) if ctx.x_is_q else [x2]
        if need_gx:
            to_save += list(w_saved) if ctx.w_is_q else [weight]
        ctx.n_x = (2 if ctx.x_is_q else 1) if need_gw else 0
        ctx.save_for_backward(*to_save)
        return y

    @staticmethod
    def backward(ctx, go: torch.Tensor):
        if ctx.plan is not None:
            gx, (gw,) = _planned_backward(ctx, [go], [ctx.N], ctx.needs_input_grad[0], [ctx.needs_input_grad[1]])
            return gx, gw if gw is None or gw.dtype == ctx.w_dtype else gw.to(ctx.w_dtype), None, None, None
        M, K, N = ctx.shapes
        saved = ctx.saved_tensors
        gx, gw = _backward_impl(
            go.reshape(M, N), ctx.config, N, ctx.x_dtype, ctx.w_dtype, saved[: ctx.n_x], saved[ctx.n_x :],
            ctx.x_is_q, ctx.w_is_q, ctx.needs_input_grad[0], ctx.needs_input_grad[1],
        )
        return gx, gw, None, None, None


def _shared_input_forward(x2, weights, c: Float8LinearConfig, scales, w_ops, need_gx: bool, need_gw: bool):
    """``ys[i] = x2 @ weights[i]^T`` with x2 quantised once.  Returns ``(ys, x_saved, w_saved)``, ``x_saved`` and each
    ``w_saved[i]`` as :func:`_forward_impl` returns them."""
    if _is_disabled(c.cast_config_input):
        return [torch.mm(x2, w.t().to(x2.dtype)) for w in weights], None, [None] * len(weights)
    share_x, share_w = _saves_quantised(c, need_gx, need_gw)
    xq, sx, x_saved, ws = _forward_operands(x2, weights, c, scales, w_ops, share_x, share_w)
    ys = ops.gemm_fp8_batch([(xq, sx, wq, sw, None, False) for wq, sw, _ in ws], out_dtype=x2.dtype)
    return ys, x_saved, [kept for _, _, kept in ws]


# Elements of the grad_outputs of linears of one input up to which they are quantised, and their products handed over, together:
# all of their float8 copies, two bytes an element, are held until then.  Beyond, one linear after the other.  Forward and backward
# of three projections with scales per row, together / one by one: 16384 x 4096 2046 / 2068 us, the backward's own peak 608 / 352 MiB,
# 16384 x 2048 834 / 843 us, 312 / 184 MiB; with one scale 2000 / 1999 and 805 / 800 us.
_MOST_TOGETHER = 256 << 20


class _Float8SharedInputMatmul(torch.autograd.Function):
    """``ys[i] = x @ W_i^T`` for several weights applied to ONE input (the q, k and v projections of an attention
    block, reference src/olmo_core/nn/attention/__init__.py:582): x is quantised once by construction, one copy of
    it is kept for all the weight gradients, and the grad_input terms are summed by the GEMM epilogues
    (``C += product``) in the order autograd adds them - the last projection's first - so outputs and gradients carry
    the bits of the modules applied one by one."""

    @staticmethod
    def forward(ctx, x2, config, n, act_dtype, *rest):
        # act_dtype: the type the modules see their input in (the autocast type when autocast is on, else x2's own).
        # Each module would convert x2 itself and autograd would add the converted-back grad_input terms in x2's type:
        # that sum is formed here when the types differ.
        weights, scales, w_ops = rest[:n], rest[n:2 * n], rest[2 * n:3 * n]
        need_gx = ctx.needs_input_grad[0]
        need_gws = [ctx.needs_input_grad[4 + i] for i in range(n)]
        ctx.set_materialize_grads(False)
        ctx.gx_dtype = x2.dtype
        if x2.dtype != act_dtype:
            x2 = x2.to(act_dtype)
        done = None
        if ctx.gx_dtype == x2.dtype and _fp8_backward(config):
            done = _planned_forward(x2, weights, config, scales, w_ops, need_gx, any(need_gws))
        ctx.plan = None
        if done is not None:
            ys, kept, ctx.plan = done
            ctx.config, ctx.M, ctx.ns, ctx.x_dtype = config, x2.shape[0], [w.shape[0] for w in weights], x2.dtype
            ctx.w_dtypes, ctx.need_gws = [w.dtype for w in weights], need_gws
            ctx.save_for_backward(kept)
            return tuple(ys)
        ys, x_saved, w_saved = _shared_input_forward(x2, weights, config, scales, w_ops, need_gx, any(need_gws))
        ctx.config = config
        ctx.x_dtype, ctx.w_dtypes = x2.dtype, [w.dtype for w in weights]
        ctx.M, ctx.ns = x2.shape[0], [w.shape[0] for w in weights]
        ctx.x_is_q, ctx.w_is_q = x_saved is not None, [k is not None for k in w_saved]
        ctx.need_gws = need_gws
        to_save = []
        if any(need_gws):
            to_save += list(x_saved) if ctx.x_is_q else [x2]
        ctx.n_x = len(to_save)
        if need_gx:
            for w, kept in zip(weights, w_saved):
                to_save += list(kept) if kept is not None else [w]
        ctx.save_for_backward(*to_save)
        return tuple(ys)

    @staticmethod
    def backward(ctx, *gos):
        n = len(ctx.ns)
        need_gx = ctx.needs_input_grad[0]
        if ctx.plan is not None:
            gx, gws = _planned_backward(ctx, gos, ctx.ns, need_gx, ctx.need_gws)
            gws = [gw if gw is None or gw.dtype == dt else gw.to(dt) for gw, dt in zip(gws, ctx.w_dtypes)]
            return (gx, None, None, None, *gws, *([None] * (2 * n)))
        saved = ctx.saved_tensors
        x_part, pos = saved[:ctx.n_x], ctx.n_x
        w_parts = []
        for i in range(n):
            k = (2 if ctx.w_is_q[i] else 1) if need_gx else 0
            w_parts.append(saved[pos:pos + k])
            pos += k
        gx, gws = None, [None] * n
        chain = ctx.gx_dtype == ctx.x_dtype  # the terms are added in the type the GEMMs write: by their epilogues
        gos = [None if go is None else go.reshape(ctx.M, ctx.ns[i]) for i, go in enumerate(gos)]
        gos = [go if go is None or go.dtype == ctx.x_dtype else go.to(ctx.x_dtype) for go in gos]
        c = ctx.config
        order = [i for i in reversed(range(n)) if gos[i] is not None]
        together = sum(gos[i].numel() for i in order) <= _MOST_TOGETHER
        made = _grad_operands(gos, c, need_gx, ctx.need_gws) if together else [None] * n
        if (order and together and chain and not _is_disabled(c.cast_config_grad_output)
                and not _is_disabled(c.cast_config_grad_output_for_grad_weight)):
            products = [_grad_input_product(gos[i], c, ctx.ns[i], made[i][0], w_parts[i], ctx.w_is_q[i], add=i != order[0])
                        for i in order if need_gx]
            wanted = [i for i in order if ctx.need_gws[i]]
            products += [_grad_weight_product(gos[i], c, made[i][1], x_part, ctx.x_is_q, ctx.w_dtypes[i]) for i in wanted]
            outs = ops.gemm_fp8_products(products, out_dtype=ctx.x_dtype)
            if need_gx:
                gx = outs.pop(0)
            for i, gw in zip(wanted, outs):
                gws[i] = gw if gw.dtype == ctx.w_dtypes[i] else gw.to(ctx.w_dtypes[i])
            return (gx, None, None, None, *gws, *([None] * (2 * n)))
        for i in reversed(range(n)):
            if gos[i] is None:
                continue
            term, gws[i] = _backward_impl(
                gos[i], ctx.config, ctx.ns[i], ctx.x_dtype, ctx.w_dtypes[i], x_part, w_parts[i],
                ctx.x_is_q, ctx.w_is_q[i], need_gx, ctx.need_gws[i], gx_into=gx if chain else None, go_operands=made[i],
            )
            if need_gx:
                gx = term if chain else (term.to(ctx.gx_dtype) if gx is None else gx.add_(term))
        return (gx, None, None, None, *gws, *([None] * (2 * n)))


def float8_projections(x: torch.Tensor, *modules: nn.Module) -> Tuple[torch.Tensor, ...]:
    """``tuple(m(x) for m in modules)`` for linear modules applied to one tensor, e.g. ``q, k, v =
    float8_projections(x, self.w_q, self.w_k, self.w_v)`` in place of the three calls at
    src/olmo_core/nn/attention/__init__.py:582.  When every module is a :class:`Float8Linear` of one config the
    input is quantised once for all of them and its gradient leaves the last grad_input GEMM already summed; outputs
    and gradients have the bits of the separate calls.  Anything else (plain ``nn.Linear``, mixed configs, a traced
    graph) is applied module by module."""
    mods = modules
    fusable = (
        len(mods) > 1 and all(isinstance(m, Float8Linear) for m in mods) and x.is_cuda
        and all(m.config is mods[0].config or m.config == mods[0].config for m in mods)
        and all(m.in_features == x.shape[-1] for m in mods) and not torch.compiler.is_compiling()
    )
    if not fusable:
        return tuple(m(x) for m in mods)
    act_dtype = torch.get_autocast_dtype(x.device.type) if torch.is_autocast_enabled() else x.dtype
    c = mods[0].config
    x2 = x.reshape(-1, x.shape[-1])
    weights = [m.weight for m in mods]
    scales = [m.precomputed_weight_scale() for m in mods]
    w_ops = [m.weight_operands() for m in mods]
    if torch.is_grad_enabled() and (x2.requires_grad or any(w.requires_grad for w in weights)):
        # (not compiling here, so nothing is to be kept from a tracer)
        ys = _Float8SharedInputMatmul.apply(x2, c, len(weights), act_dtype, *weights, *scales, *w_ops)
    else:
        ys = _shared_input_forward(x2.to(act_dtype), weights, c, scales, w_ops, False, False)[0]
    outs = []
    for m, y in zip(mods, ys):
        if x.dim() != 2:
            y = y.reshape(*x.shape[:-1], y.shape[1])
        bias = m.bias
        outs.append(y if bias is None else y + bias.to(y.dtype))
    return tuple(outs)


# Operator arguments must be plain values: under torch.compile a config travels as its index in this list.  Configs
# are registered when a module is built (tracing must not mutate the list).
_COMPILED_CONFIGS: list = []

# Likewise the modules (as weak references): a compiled call names its module by index, and the operator, which runs
# eagerly, asks that module for its precomputed weight scale and kept float8 weight copies - lookups by address and
# version counter that a traced graph cannot contain.
_COMPILED_MODULES: list = []


def _register_module(m) -> int:
    import weakref

    _COMPILED_MODULES.append(weakref.ref(m))
    return len(_COMPILED_MODULES) - 1


def _kept_weight_state(module_id: int, weight: torch.Tensor):
    """``(precomputed scale, kept operands)`` of the registered module if ``weight`` is that module's weight."""
    if module_id < 0 or module_id >= len(_COMPILED_MODULES):
        return None, None
    m = _COMPILED_MODULES[module_id]()
    if m is None or m.weight.data_ptr() != weight.data_ptr() or m.weight.shape != weight.shape:
        return None, None
    return m.precomputed_weight_scale(), m.weight_operands()


def _register_config(c: Float8LinearConfig) -> int:
    idx = getattr(c, "_compiled_id", None)
    if idx is None:
        _COMPILED_CONFIGS.append(c)
        idx = len(_COMPILED_CONFIGS) - 1
        c._compiled_id = idx
    return idx


@torch.compiler.disable
def _eager_matmul(x2, weight, config, weight_scale, weight_ops=None):
    return _Float8Matmul.apply(x2, weight, config, weight_scale, weight_ops)


def float8_linear_function(
    x: torch.Tensor, weight: torch.Tensor, config: Float8LinearConfig, weight_scale: Optional[torch.Tensor] = None,
    weight_ops: Optional[Tuple[torch.Tensor, torch.Tensor, torch.Tensor]] = None, module_id: int = -1,
) -> torch.Tensor:
    """``x [*, K] @ weight[N, K].T`` through the float8 path, differentiable in x and weight.

    ``weight_scale``: a precomputed tensorwise scale of ``weight`` (float32 ``[1]``), used instead of reducing the
    weight's amax again; ignored unless the weight cast is tensorwise.
    ``weight_ops``: float8 copies of ``weight`` made earlier (``(q [N, K], q_t [K, pad16(N)], scale [1])``, as
    :meth:`Float8Linear.weight_operands` returns them), used instead of quantising ``weight`` again; eager only.

    Under ``torch.compile`` the call becomes a pair of registered custom operators (forward, backward) with shape
    functions, so a compiled block keeps one graph; eagerly it is an ordinary ``autograd.Function``.
    """
    K = x.shape[-1]
    if weight.dim() != 2 or weight.shape[1] != K:
        raise ValueError(f"float8 linear: input features {K} do not match weight {tuple(weight.shape)}")
    x2 = x if x.dim() == 2 else x.reshape(-1, K)
    cfg_id = getattr(config, "_compiled_id", -1)
    compiling = torch.compiler.is_compiling()
    if compiling and cfg_id >= 0:
        from . import compiled

        y = compiled.linear(x2, weight, cfg_id, weight_scale, module_id)
    elif not compiling and not (torch.is_grad_enabled() and (x2.requires_grad or weight.requires_grad)):
        # nothing to differentiate (evaluation, generation): no autograd node, nothing kept for a backward
        done = None if _is_disabled(config.cast_config_input) else _planned_forward(x2, (weight,), config, (weight_scale,), (weight_ops,), False, False)
        y = done[0][0] if done is not None else _forward_impl(x2, weight, config, weight_scale, False, False, weight_ops)[0]
    elif not compiling:
        y = _Float8Matmul.apply(x2, weight, config, weight_scale, weight_ops)
    else:  # a config no module registered: a graph break
        y = _eager_matmul(x2, weight, config, weight_scale, weight_ops)
    return y if x.dim() == 2 else y.reshape(*x.shape[:-1], weight.shape[0])


class Float8Linear(nn.Linear):
    """
    Drop-in ``nn.Linear`` whose forward / backward matmuls run in float8 with dynamic scaling.
    Use :meth:`from_float` (or :func:`convert_to_float8_training`) to create it from an existing module.
    """

    def __init__(self, *args, config: Optional[Float8LinearConfig] = None, **kwargs):
        super().__init__(*args, **kwargs)
        self.config = config if config is not None else Float8LinearConfig()
        self._bind_config()

    def _bind_config(self) -> None:
        c = self.config
        _register_config(c)
        self._module_id = _register_module(self)
        self.scaling_type_input = c.cast_config_input.scaling_type
        self.scaling_type_weight = c.cast_config_weight.scaling_type
        self.scaling_type_grad_output = c.cast_config_grad_output.scaling_type

    def forward(self, input: torch.Tensor) -> torch.Tensor:
        if torch.is_autocast_enabled():
            input = input.to(torch.get_autocast_dtype(input.device.type))
        # (the stored scale is checked against the weight's address and version counter: not traceable)
        compiling = torch.compiler.is_compiling()
        scale = None if compiling else self.precomputed_weight_scale()
        w_ops = None if compiling else self.weight_operands()
        out = float8_linear_function(input, self.weight, self.config, scale, w_ops, self._module_id)
        bias = self.bias
        if bias is not None:
            out = out + bias.to(out.dtype)
        return out

    def precomputed_weight_scale(self) -> Optional[torch.Tensor]:
        """The scale stored by :func:`precompute_float8_dynamic_scale_for_fsdp` if the weight has not been
        modified (or replaced) since; ``None`` otherwise, and the forward then reduces the amax itself."""
        entry = getattr(self, "_precomputed_weight_scale", None)
        if entry is None:
            return None
        scale, ptr, version = entry
        w = self.weight
        if w.is_inference():  # (inference tensors have no version counter)
            return None
        if w.data_ptr() != ptr or w._version != version or not _is_tensorwise(self.config.cast_config_weight):
            return None
        return scale

    def weight_operands(self) -> Optional[Tuple[torch.Tensor, torch.Tensor, torch.Tensor]]:
        """Float8 copies of the weight that outlive one call: ``(q [N, K], q_t [K, pad16(N)], scale [1])``, made
        on first use and kept until the weight is modified or replaced (address and version counter), so that
        the micro-batches of one optimizer step, or the steps of a generation loop, quantise each weight once.

        Only with ``config.enable_fsdp_float8_all_gather``: upstream that switch makes FSDP hold and communicate
        the float8 weight (computed from the precomputed scale, ``src/olmo_core/float8/__init__.py:54-62``,
        ``src/olmo_core/float8/ao.py:173-180``); on one device what remains of it is that the float8 weight is
        materialised once per weight update rather than once per forward.  Costs two bytes per parameter.
        ``None`` when the switch is off, the weight is not a contiguous GPU tensor, or forward and grad_input
        quantise the weight differently.  Bytes and scale equal those a forward would make itself.  (A write
        through ``weight.data`` moves no version counter and goes unnoticed, as for the precomputed scales;
        :func:`precompute_float8_dynamic_scale_for_fsdp` drops the copies.)"""
        c = self.config
        if not c.enable_fsdp_float8_all_gather:
            return None
        w = self.weight
        if not _shared_tensorwise(c.cast_config_weight, c.cast_config_weight_for_grad_input):
            return None
        if not w.is_cuda or not w.is_contiguous() or w.dtype not in (torch.bfloat16, torch.float32) or w.is_inference():
            return None
        key = (w.data_ptr(), w._version, w.dtype, tuple(w.shape))
        entry = getattr(self, "_weight_operands", None)
        if entry is not None and entry[0] == key:
            return entry[1]
        with torch.no_grad():
            made = ops.cast_tensorwise(
                w.detach(), c.cast_config_weight.target_dtype, pow2=c.round_scales_to_power_of_2,
                want_rowmajor=True, want_transposed=True, scale=self.precomputed_weight_scale(),
            )
        self._weight_operands = (key, made)
        return made

    def extra_repr(self) -> str:
        c = self.config
        parts = [
            f"i:{c.cast_config_input.short_str()}",
            f"w:{c.cast_config_weight.short_str()}",
            f"go:{c.cast_config_grad_output.short_str()}",
        ]
        if c.cast_config_input_for_grad_weight != c.cast_config_input:
            parts.append(f"i_gw:{c.cast_config_input_for_grad_weight.short_str()}")
        if c.cast_config_weight_for_grad_input != c.cast_config_weight:
            parts.append(f"w_gi:{c.cast_config_weight_for_grad_input.short_str()}")
        if c.cast_config_grad_output_for_grad_weight != c.cast_config_grad_output:
            parts.append(f"go_gw:{c.cast_config_grad_output_for_grad_weight.short_str()}")
        return f'{super().extra_repr()}, cast_configs={",".join(parts)}'

    @classmethod
    def from_float(cls, mod: nn.Linear, config: Optional[Float8LinearConfig] = None) -> "Float8Linear":
        """New module sharing ``mod``'s Parameters; reads no weight values (works on the meta device)."""
        config = config if config is not None else Float8LinearConfig()
        if config.emulate:
            raise NotImplementedError(
                "emulate=True selects a CPU-emulated matmul upstream; this library only has the native gfx950 path"
            )
        config.check_gemm_operands()
        with torch.device("meta"):
            new = cls(mod.in_features, mod.out_features, bias=False, config=config)
        new.weight = mod.weight
        new.bias = mod.bias
        return new


def _swap(
    module: nn.Module,
    make: Callable[[nn.Linear], nn.Module],
    module_filter_fn: Optional[Callable[[nn.Module, str], bool]],
) -> nn.Module:
    """Post-order walk replacing every ``nn.Linear`` the filter accepts; the filter sees only Linears."""
    if isinstance(module, nn.Linear) and (module_filter_fn is None or module_filter_fn(module, "")):
        if len(list(module.children())) > 0:
            raise AssertionError(f"Does not support a root nn.Linear with children: {module}")
        return make(module)

    visited = set()

    def walk(m: nn.Module, fqn: str, parent: Optional[nn.Module], name: Optional[str]) -> None:
        if id(m) in visited:
            return
        visited.add(id(m))
        for child_name, child in list(m.named_children()):
            walk(child, f"{fqn}.{child_name}" if fqn else child_name, m, child_name)
        if parent is not None and isinstance(m, nn.Linear) and not isinstance(m, Float8Linear):
            if module_filter_fn is None or module_filter_fn(m, fqn):
                setattr(parent, name, make(m))

    walk(module, "", None, None)
    return module


def convert_to_float8_training(
    module: nn.Module,
    *,
    module_filter_fn: Optional[Callable[[nn.Module, str], bool]] = None,
    config: Optional[Float8LinearConfig] = None,
) -> nn.Module:
    """
    Swap ``nn.Linear`` modules for :class:`Float8Linear` in place and return the (possibly new) root.
    ``module_filter_fn(mod, fqn)`` is consulted for Linear modules only; returning False keeps the module.
    """
    config = config if config is not None else Float8LinearConfig()
    return _swap(module, lambda m: Float8Linear.from_float(m, config), module_filter_fn)


def precompute_float8_dynamic_scale_for_fsdp(module: nn.Module) -> None:
    """
    Refresh the tensorwise weight scales of every :class:`Float8Linear` under ``module`` in one batch of kernel
    launches; call it right after the optimizer step (reference: torchao's function of the same name, called
    from ``src/olmo_core/nn/transformer/model.py:1001-1008``).  Forwards then skip the weight's amax pass until
    the weight changes again; the scales are the ones the forward would compute itself, bit for bit.
    """
    groups: dict = {}
    for m in module.modules():
        if not isinstance(m, Float8Linear):
            continue
        m._precomputed_weight_scale = None
        m._weight_operands = None
        c = m.config
        w = m.weight
        if not _is_tensorwise(c.cast_config_weight) or not w.is_cuda or not w.is_contiguous():
            continue
        if w.dtype not in (torch.bfloat16, torch.float32) or w.data_ptr() % 16:
            continue
        key = (w.device, w.dtype, c.cast_config_weight.target_dtype, c.round_scales_to_power_of_2)
        groups.setdefault(key, []).append(m)
    for (_, _, fp8_dtype, pow2), mods in groups.items():
        for start in range(0, len(mods), 65535):
            chunk = mods[start:start + 65535]
            with torch.no_grad():
                scales = ops.multi_tensor_scales([m.weight.detach() for m in chunk], fp8_dtype, pow2=pow2)
            for i, m in enumerate(chunk):
                m._precomputed_weight_scale = (scales[i:i + 1], m.weight.data_ptr(), m.weight._version)
