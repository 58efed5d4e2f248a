"""
SwiGLU feed-forward block: the host of the float8 linears in the dense models
(reference: src/olmo_core/nn/feed_forward.py:142-171, ``w2(silu(w1(x)) * w3(x))``; flops convention
:206-209).  The three projections are ordinary ``nn.Linear`` modules so that
``Float8Config.apply_float8_linear`` swaps them.

When all three are tensorwise ``Float8Linear`` modules without bias the block runs as one autograd function
that performs exactly the casts and GEMMs the three modules would perform one by one (same bytes, same scales,
same outputs), but quantises ``x`` once for ``w1`` and ``w3``, takes the amax of ``h`` and of the two gate
gradients inside the SwiGLU kernels that produce them (no separate pass over the largest tensors), and saves
fp8 copies instead of the bf16 activations ``x`` and ``h``.
"""

from __future__ import annotations

import torch
import torch.nn as nn

from ..float8 import ops, plan
from ..float8.linear import Float8Linear, _shared_tensorwise, needs_autograd

__all__ = ["FeedForward", "swiglu"]

# Test hook: when set to a dict, the fused function stores clones of its bf16 intermediates (x1, x3, h, gh) there,
# so that a checker can feed each stage's actual input to a reference of that stage, together with the float8
# operands it made of h, g1 and g3 and their scales (sh, hq, sg1, g1q, sg3, g3q): what the GEMMs actually consumed.
STAGE_SINK = None

# Run the two input projections and the SwiGLU between them as one launch where the shape allows (same bits as the
# three separate launches); a switch so that the two routes can be compared.
FUSE_SWIGLU_EPILOGUE = True

# Take the amax of the two gate gradients from the row-segment codes that the fused forward launch and the GEMM that
# produces grad_h record (same bits as the pass over gh, x1 and x3 it replaces); a switch so that the two routes can be
# compared.
SWIGLU_AMAX_FROM_CODES = True


class _SwiGLU(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x1: torch.Tensor, x3: torch.Tensor):
        h, _ = ops.swiglu_fwd(x1, x3, want_amax=False)
        ctx.save_for_backward(x1, x3)
        return h

    @staticmethod
    def backward(ctx, gh: torch.Tensor):
        x1, x3 = ctx.saved_tensors
        g1, g3, _, _ = ops.swiglu_bwd(x1, x3, gh, want_amax=False)
        return g1, g3


@torch.compiler.disable
def swiglu(x1: torch.Tensor, x3: torch.Tensor) -> torch.Tensor:
    """``silu(x1) * x3`` for bfloat16 GPU tensors (one fused kernel forward, one backward)."""
    return _SwiGLU.apply(x1, x3)


def _use_codes(M: int, D: int, H: int, any_grad: bool) -> bool:
    """Whether the fused forward launch records the row-segment codes of x1 and x3 for the backward pass."""
    return any_grad and SWIGLU_AMAX_FROM_CODES and H % 64 == 0 and ops.gemm_codes_supported(M, H, D)


def _fused_launch_ok(M: int, D: int, H: int) -> bool:
    return FUSE_SWIGLU_EPILOGUE and ops.swiglu_gemm_pays(M, H, D)


def _mlp_forward(x, w1, w2, w3, c, need, ws=(None, None, None), wo=(None, None, None), keep=True):
    """y = (silu(x W1^T) * (x W3^T)) W2^T with tensorwise float8 GEMMs; x [M, D], W1/W3 [H, D], W2 [D, H].  x is
    converted to bfloat16 first if it is of another type (float32 activations under autocast: each of the three
    modules would convert its own input).
    need: which of (x, w1, w2, w3) get a gradient.  ws: weight scales precomputed after the optimizer step (None: reduce
    the amax here); wo: float8 copies the modules keep between calls (None: quantise the weight here); both in the
    order (w1, w2, w3).  Returns ``(y, saved)``, ``saved`` being the 13 tensors :func:`_mlp_backward` takes (an empty
    tensor where nothing is kept).  keep=False: only ``y`` is wanted (no gradients, ``saved`` is not to be used)."""
    pow2 = c.round_scales_to_power_of_2
    in_dt, w_dt = c.cast_config_input.target_dtype, c.cast_config_weight.target_dtype
    any_grad = any(need)
    ws1, ws2, ws3 = ws
    wo1, wo2, wo3 = wo
    x_codes = None
    if x.dtype != torch.bfloat16:
        x = x.to(torch.bfloat16)
    M, D, H = x.shape[0], x.shape[1], w1.shape[0]
    # a generation step: launches that wait for one another are the time, so the activations are quantised by the GEMMs
    few_rows = not keep and STAGE_SINK is None and ops.few_rows_supported(M, H, in_dt, w_dt) and w2.shape[0] % 8 == 0
    x_in_gemm = few_rows and ops.few_rows_quantises(M, D)
    # x and every weight that has no float8 copy yet are quantised together: one launch for the maxima, one for the casts
    items = [] if x_in_gemm else [(x, dict(want_transposed=need[1] or need[3], whole_steps=True))]
    items += [(w, dict(want_transposed=t, scale=s))
              for w, t, s, o in ((w1, need[0], ws1, wo1), (w3, need[0], ws3, wo3), (w2, any_grad, ws2, wo2)) if o is None]
    if in_dt == w_dt:
        made = iter(ops.cast_tensorwise_batch(items, in_dt, pow2=pow2) if items else ())
    else:
        made = iter([ops.cast_tensorwise(t, in_dt if t is x else w_dt, pow2=pow2, **kw) for t, kw in items])
    xq, xq_t, sx = (x, None, None) if x_in_gemm else next(made)
    w1q, w1q_t, s1 = wo1 or next(made)
    w3q, w3q_t, s3 = wo3 or next(made)
    w2q, w2q_t, s2 = wo2 or next(made)
    if few_rows:
        h, h_slots = ops.few_rows_swiglu(xq, sx, w1q, s1, w3q, s3, pow2=pow2)
        if ops.few_rows_quantises(M, H, have_slots=True):
            return ops.few_rows_cast_gemm(h, h_slots, w2q, s2, pow2=pow2), ()
        hq, _, sh = ops.cast_tensorwise(h, in_dt, pow2=pow2, slots=h_slots)
        return ops.gemm_fp8(hq, sh, w2q, s2, out_dtype=x.dtype), ()
    if _fused_launch_ok(M, D, H):
        # both input projections and the activation in one launch: x1 and x3 are never read back
        if _use_codes(M, D, H, any_grad):
            x1, x3, h, h_slots, x_codes = ops.gemm_fp8_swiglu(xq, sx, w1q, s1, w3q, s3, want_codes=True)
        else:
            x1, x3, h, h_slots = ops.gemm_fp8_swiglu(xq, sx, w1q, s1, w3q, s3)
    else:
        x1, x3 = ops.gemm_fp8_batch([(xq, sx, w1q, s1, None, False), (xq, sx, w3q, s3, None, False)], out_dtype=x.dtype)
        h, h_slots = ops.swiglu_fwd(x1, x3, want_amax=True)
    if STAGE_SINK is not None:
        STAGE_SINK.update(x1=x1.clone(), x3=x3.clone(), h=h.clone())
    hq, hq_t, sh = ops.cast_tensorwise(h, in_dt, pow2=pow2, want_transposed=need[2], slots=h_slots, whole_steps=True)
    if STAGE_SINK is not None:
        STAGE_SINK.update(sh=sh.clone(), hq=hq.clone())
    y = ops.gemm_fp8(hq, sh, w2q, s2, out_dtype=x.dtype)
    opt = lambda t: t if t is not None else x.new_empty(0)  # noqa: E731
    saved = (opt(xq_t), sx, x1, x3, opt(hq_t), sh, opt(w1q_t), s1, opt(w2q_t), s2, opt(w3q_t), s3, opt(x_codes))
    return y, saved


def _mlp_backward(gy, saved, c, dims, dtypes, need):
    """The four gradients ``(gx, gw1, gw2, gw3)`` (``None`` where not needed) of :func:`_mlp_forward`.  dtypes: of the
    x the forward was given and of the three weights.  For a bfloat16 x the two grad_x terms are added by the second
    GEMM's epilogue; for an x of another type they are added in that type, as autograd adds the converted-back
    gradients of the two modules that each converted x."""
    xq_t, sx, x1, x3, hq_t, sh, w1q_t, s1, w2q_t, s2, w3q_t, s3, x_codes = saved
    pow2 = c.round_scales_to_power_of_2
    go_dt = c.cast_config_grad_output.target_dtype
    gx_dt, w1_dt, w2_dt, w3_dt = dtypes
    x_dt = torch.bfloat16
    M, D, H = dims
    need_x, need_w1, need_w2, need_w3 = need
    gy = gy.reshape(M, D)
    if gy.dtype != x_dt:
        gy = gy.to(x_dt)
    need_gh = need_x or need_w1 or need_w3
    gyq, gyq_t, sgy = ops.cast_tensorwise(gy, go_dt, pow2=pow2, want_rowmajor=need_gh, want_transposed=need_w2,
                                           whole_steps=True)
    # (the weights' gradients leave the GEMMs in the weights' type: float32 that holds the bf16 values under autocast)
    w2_product = (gyq_t, sgy, hq_t, sh, None, False, w2_dt)
    gx = gw1 = gw2 = gw3 = None
    if need_w2 and not need_gh:
        (gw2,) = ops.gemm_fp8_batch([w2_product], out_dtype=x_dt)
    if need_gh:
        # g1 and g3 are needed in fp8 only, and their tensorwise scales need the amax of both first.  Where the
        # forward recorded the row-segment codes of x1 and x3, the GEMM that produces gh records those of gh, and the
        # amax follows by computing a small share of the segments; otherwise a pass over the three tensors takes it.
        codes = None
        if x_codes.numel() and x_dt == torch.bfloat16 and ops.gemm_codes_supported(M, H, D):
            if need_w2:
                (gw2,) = ops.gemm_fp8_batch([w2_product], out_dtype=x_dt)
            gh, gh_codes = ops.gemm_fp8_codes(gyq, sgy, w2q_t, s2, k=D)
            codes = (gh_codes, x_codes)
        else:
            gh, *rest = ops.gemm_fp8_products([(gyq, sgy, w2q_t, s2, D, False)] + ([w2_product] if need_w2 else []), out_dtype=x_dt)
            gw2 = rest[0] if need_w2 else None
        if STAGE_SINK is not None:
            STAGE_SINK.update(gh=gh.clone())
        need_t = need_w1 or need_w3
        # then the recompute-and-cast pass (no bf16 round trip of g1, g3)
        g1q, g1q_t, sg1, g3q, g3q_t, sg3 = ops.swiglu_bwd_cast(
            x1, x3, gh, go_dt, pow2=pow2, want_rowmajor=need_x, want_transposed=need_t, codes=codes, whole_steps=True)
        del gh
        if STAGE_SINK is not None:
            STAGE_SINK.update(sg1=sg1.clone(), sg3=sg3.clone(), amax_from_codes=codes is not None,
                              g1q=None if g1q is None else g1q.clone(), g3q=None if g3q is None else g3q.clone())
        products = []
        if need_x and gx_dt == x_dt:
            # the sum of the two halves as autograd forms it (two bf16 tensors added), by the second GEMM's epilogue
            products += [(g1q, sg1, w1q_t, s1, H, False), (g3q, sg3, w3q_t, s3, H, True)]
        elif need_x:
            products += [(g3q, sg3, w3q_t, s3, H, False), (g1q, sg1, w1q_t, s1, H, False)]
        if need_w1:
            products.append((g1q_t, sg1, xq_t, sx, None, False, w1_dt))
        if need_w3:
            products.append((g3q_t, sg3, xq_t, sx, None, False, w3_dt))
        outs = ops.gemm_fp8_products(products, out_dtype=x_dt)
        if need_w3:
            gw3 = outs.pop()
        if need_w1:
            gw1 = outs.pop()
        if need_x and gx_dt == x_dt:
            gx = outs[0]
        elif need_x:
            # (autograd runs w3's backward first: its term is the one the other is added to)
            gx = outs[0].to(gx_dt)
            gx.add_(outs[1])

    def as_param(g, dt):
        return g if g is None or g.dtype == dt else g.to(dt)

    return gx, as_param(gw1, w1_dt), as_param(gw2, w2_dt), as_param(gw3, w3_dt)


def _planned_forward(x, weights, c, need, ws, wo, keep: bool):
    """:func:`_mlp_forward` from a plan: ``([y], kept, plan)`` or ``None``."""
    if STAGE_SINK is not None or x.dtype != torch.bfloat16 or (keep and any(o is not None for o in wo)):
        return None  # (a conversion of x, and kept weights among what the backward takes, are not recorded)
    pow2 = c.round_scales_to_power_of_2
    options = ("mlp", need, keep, pow2, c.cast_config_input.target_dtype, c.cast_config_weight.target_dtype,
               c.cast_config_grad_output.target_dtype, FUSE_SWIGLU_EPILOGUE, SWIGLU_AMAX_FROM_CODES)

    def recorded(px, p1, p2, p3, *rest):
        given = tuple(rest[3 + 3 * i:6 + 3 * i] if rest[3 + 3 * i] is not None else None for i in range(3))
        y, saved = _mlp_forward(px, p1, p2, p3, c, need, rest[:3], given, keep)
        return [y], saved if keep else None

    if None not in wo and not keep:  # generation: what is needed of three weights are their row-major float8 copies

        def kept_weights(px, q1, q2, q3, t1, t2, t3):
            return [_mlp_forward(px, q1, q2, q3, c, need, (None,) * 3, ((q1, None, t1), (q2, None, t2), (q3, None, t3)), False)[0]], None

        return plan.call(kept_weights, [x, *(o[0] for o in wo), *(o[2] for o in wo)], options, own=6)
    inputs = [x, *weights, *ws]
    for o in wo:
        inputs += (None, None, None) if o is None else o
    return plan.call(recorded, inputs, options, own=9)


class _Float8SwiGLUMLP(torch.autograd.Function):
    """The fused block as an eager autograd function (a traced graph takes the registered operators of
    ``olmo_core_amd.float8.compiled`` instead, which run the same two routines)."""

    @staticmethod
    def forward(ctx, x, w1, w2, w3, config, ws1=None, ws2=None, ws3=None, wo1=None, wo2=None, wo3=None):
        need = tuple(ctx.needs_input_grad[:4])
        done = _planned_forward(x, (w1, w2, w3), config, need, (ws1, ws2, ws3), (wo1, wo2, wo3), True)
        ctx.plan = None
        if done is not None:
            (y,), kept, ctx.plan = done
            saved = (kept,)
        else:
            y, saved = _mlp_forward(x, w1, w2, w3, config, need, (ws1, ws2, ws3), (wo1, wo2, wo3))
        ctx.config = config
        ctx.dtypes = (x.dtype, w1.dtype, w2.dtype, w3.dtype)
        ctx.dims = (x.shape[0], x.shape[1], w1.shape[0])
        ctx.save_for_backward(*saved)
        return y

    @staticmethod
    def backward(ctx, gy):
        need = tuple(ctx.needs_input_grad[:4])
        if ctx.plan is None:
            return _mlp_backward(gy, ctx.saved_tensors, ctx.config, ctx.dims, ctx.dtypes, need) + (None,) * 7
        (kept,), bf16 = ctx.saved_tensors, torch.bfloat16
        done = None
        if STAGE_SINK is None and ctx.dtypes[0] == bf16:
            if gy.dtype != bf16 or not gy.is_contiguous():
                gy = gy.to(bf16).contiguous()

            def recorded(slab, pgy):
                grads = _mlp_backward(pgy, ctx.plan.saved_places(slab), ctx.config, ctx.dims, ctx.dtypes, need)
                return [g for g in grads if g is not None], None

            done = plan.call(recorded, [kept, gy], ("backward", need), within=ctx.plan)  # (the forward's plan knows the types)
        if done is None:
            return _mlp_backward(gy, ctx.plan.saved_tensors(kept), ctx.config, ctx.dims, ctx.dtypes, need) + (None,) * 7
        grads = iter(done[0])
        return (*(next(grads) if n else None for n in need), *(None,) * 7)


def _fusable_modules(ff: "FeedForward", same_object: bool = False) -> bool:
    """The three projections are float8 modules of one tensorwise config without bias.  same_object: only accept one
    shared config object (what a model conversion hands to every module), without comparing configs field by field:
    the form a traced graph evaluates."""
    return ff.fuse_float8 and _fusable((ff.w1, ff.w2, ff.w3), same_object)


def _fusable(mods, same_object: bool = False) -> bool:
    for m in mods:
        if not isinstance(m, Float8Linear) or m.bias is not None:
            return False
    c = mods[0].config
    for m in mods[1:]:
        if m.config is not c and (same_object or m.config != c):
            return False
    return (
        _shared_tensorwise(c.cast_config_input, c.cast_config_input_for_grad_weight)
        and _shared_tensorwise(c.cast_config_weight, c.cast_config_weight_for_grad_input)
        and _shared_tensorwise(c.cast_config_grad_output, c.cast_config_grad_output_for_grad_weight)
    )


class FeedForward(nn.Module):
    """Gated feed-forward with SiLU activation: ``w2(silu(w1 x) * w3 x)``."""

    def __init__(
        self,
        *,
        d_model: int,
        hidden_size: int,
        bias: bool = True,
        dtype: torch.dtype = torch.float32,
        init_device: str = "cpu",
        fuse_float8: bool = True,
    ):
        super().__init__()
        self.d_model = d_model
        self.hidden_size = hidden_size
        self.fuse_float8 = fuse_float8
        self.w1 = nn.Linear(d_model, hidden_size, bias=bias, dtype=dtype, device=init_device)
        self.w2 = nn.Linear(hidden_size, d_model, bias=bias, dtype=dtype, device=init_device)
        self.w3 = nn.Linear(d_model, hidden_size, bias=bias, dtype=dtype, device=init_device)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        # The fused block does what the three modules do one by one, including their first step under autocast (the
        # input goes to the autocast type: src/olmo_core/train/train_module/transformer/train_module.py:593-597 runs the
        # model that way); it takes bfloat16 activations on the GPU.
        compiling = torch.compiler.is_compiling()
        act_dtype = torch.get_autocast_dtype("cuda") if x.is_cuda and torch.is_autocast_enabled() else x.dtype
        xa = x  # (the conversion to the autocast type happens inside the fused function)
        if compiling:
            # a traced graph (the reference compiles every block, src/olmo_core/nn/transformer/block.py:78-79) keeps the
            # fused launches: the block is one registered operator with a shape function
            cfg_id = getattr(self.w1.config, "_compiled_id", -1) if _fusable_modules(self, same_object=True) else -1
            if cfg_id >= 0 and xa.is_cuda and act_dtype == torch.bfloat16:
                from ..float8 import compiled

                x2 = xa.reshape(-1, xa.shape[-1])
                y = compiled.swiglu_mlp(x2, self.w1.weight, self.w2.weight, self.w3.weight, cfg_id,
                                        (self.w1._module_id, self.w2._module_id, self.w3._module_id))
                return y.reshape(*x.shape[:-1], self.w2.weight.shape[0])
        elif xa.is_cuda and act_dtype == torch.bfloat16 and self.fuse_float8 and _fusable(mods := (self.w1, self.w2, self.w3)):
            x2 = xa if xa.dim() == 2 else xa.reshape(-1, xa.shape[-1])
            c = mods[0].config
            weights = tuple(m.weight for m in mods)
            scales = tuple(m.precomputed_weight_scale() for m in mods)
            operands = tuple(m.weight_operands() for m in mods)
            if needs_autograd(x2, *weights):
                y = _Float8SwiGLUMLP.apply(x2, *weights, c, *scales, *operands)  # (not compiling: no tracer to keep it from)
            else:
                # nothing to differentiate: no transposed float8 copies, nothing kept for a backward (an autograd
                # function reports its inputs' requires_grad also where gradients are off)
                done = _planned_forward(x2, weights, c, (False,) * 4, scales, operands, False)
                y = done[0][0] if done is not None else _mlp_forward(x2, *weights, c, (False,) * 4, scales, operands, keep=False)[0]
            return y if xa.dim() == 2 else y.reshape(*x.shape[:-1], y.shape[1])
        x1, x3 = self.w1(x), self.w3(x)
        if x1.is_cuda and x1.dtype == torch.bfloat16 and not compiling:
            h = swiglu(x1, x3)
        else:
            h = torch.nn.functional.silu(x1) * x3
        return self.w2(h)

    def num_flops_per_token(self, seq_len: int) -> int:
        del seq_len
        return 6 * sum(p.numel() for p in self.parameters())
