"""
The work that users of this package have it do, as measurable cases.

Every case goes through the public entry points (``Float8Config.apply_float8_linear`` on a model, then the model's own
calls) and belongs to one of five kinds:

* ``mlp_fwd``    evaluation and generation through a SwiGLU feed-forward block whose float8 weights are kept
                 (``AOFloat8LinearConfig.recommended()``): decode at a few tokens, prefill at hundreds to thousands
* ``linear_fwd`` one float8 projection without gradients, the weight quantised by every call (the plain recipes)
* ``mlp_train``  forward and backward of the feed-forward block, bfloat16 parameters or float32 ones under autocast
* ``attn_train`` forward and backward of the q, k, v and output projections of an attention block, all three recipes
* ``moe_train``, ``moe_fwd``  the routed dropless-MoE layer: training, and evaluation / generation with kept weights

:func:`listed` names twelve of them, :func:`draw` gives others of the same ranges.
"""

import math

import torch

from olmo_core_amd.float8 import AOFloat8LinearConfig, AOFloat8LinearRecipe, Float8Config
from olmo_core_amd.float8.linear import float8_projections
from olmo_core_amd.nn import DroplessMoEMLP, FeedForward, ParallelDroplessMLP

# (d_model, hidden) of feed-forward blocks: small generic ones, one whose sizes are multiples of 16 and of nothing
# larger, the 7B and the 32B shape
_MLP_DIMS = [(768, 2048), (1024, 2816), (1040, 2768), (2048, 8192), (4096, 11008), (5120, 27648)]
# (in, out) of single projections
_LINEAR_DIMS = [(1024, 1024), (1024, 2816), (1040, 2768), (2048, 8192), (4096, 4096), (4096, 11008), (11008, 4096)]
_ATTN_DIMS = [768, 1024, 2048, 4096]
# (d_model, expert hidden, experts, top_k)
_MOE_DIMS = [(512, 256, 8, 2), (1024, 512, 32, 4), (1024, 1792, 8, 2), (2048, 1024, 64, 8)]
_RECIPES = ["tensorwise", "rowwise", "rowwise_with_gw_hp"]

# no drawn case has more arithmetic than the largest listed one
_MOST_FLOPS = 18.0 * 8192 * 5120 * 27648


def listed():
    return [
        # one sequence generating: every layer's block is called on a single token, where launches and host work count
        {"name": "mlp_decode_1", "kind": "mlp_fwd", "tokens": 1, "d": 4096, "h": 11008},
        # a batch of sequences generating, an odd number of them in flight
        {"name": "mlp_decode_23", "kind": "mlp_fwd", "tokens": 23, "d": 4096, "h": 11008},
        # a prompt of ordinary length
        {"name": "mlp_prefill_777", "kind": "mlp_fwd", "tokens": 777, "d": 4096, "h": 11008},
        # one projection in evaluation, its weight quantised by the call
        {"name": "linear_fwd_2048", "kind": "linear_fwd", "tokens": 2048, "d": 4096, "n": 11008, "recipe": "tensorwise"},
        # a small model in training, the token count of a packed batch (not a multiple of anything)
        {"name": "mlp_train_small", "kind": "mlp_train", "tokens": 1999, "d": 1024, "h": 2816, "autocast": False, "outliers": False},
        # float32 parameters under bfloat16 autocast, as the trainer runs a model without sharding
        {"name": "mlp_train_autocast", "kind": "mlp_train", "tokens": 4096, "d": 2048, "h": 8192, "autocast": True, "outliers": False},
        # the 7B block at batch 4 x 4096
        {"name": "mlp_train_7b", "kind": "mlp_train", "tokens": 16384, "d": 4096, "h": 11008, "autocast": False, "outliers": False},
        # the 32B block, activations with outliers: the largest case
        {"name": "mlp_train_32b", "kind": "mlp_train", "tokens": 8192, "d": 5120, "h": 27648, "autocast": False, "outliers": True},
        # attention projections of the 7B shape, per-row scales
        {"name": "attn_train_7b", "kind": "attn_train", "tokens": 16384, "d": 4096, "recipe": "rowwise"},
        # the same of a smaller model on a ragged batch
        {"name": "attn_train_ragged", "kind": "attn_train", "tokens": 1537, "d": 2048, "recipe": "rowwise"},
        # a routed expert layer in training: 64 experts of skewed popularity, some of them empty
        {"name": "moe_train", "kind": "moe_train", "tokens": 16384, "d": 2048, "h": 1024, "experts": 64, "top_k": 8},
        # the same layer generating for a small batch of sequences
        {"name": "moe_decode_48", "kind": "moe_fwd", "tokens": 48, "d": 2048, "h": 1024, "experts": 64, "top_k": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(["mlp_fwd", "mlp_fwd", "linear_fwd", "mlp_train", "mlp_train", "attn_train", "moe_train", "moe_fwd"])
        if kind == "mlp_fwd":
            d, h = rng.choice(_MLP_DIMS)
            case = {"kind": kind, "tokens": _log_int(rng, 1, 8192), "d": d, "h": h}
        elif kind == "linear_fwd":
            d, n = rng.choice(_LINEAR_DIMS)
            case = {"kind": kind, "tokens": _log_int(rng, 1, 8192), "d": d, "n": n, "recipe": rng.choice(_RECIPES)}
        elif kind == "mlp_train":
            d, h = rng.choice(_MLP_DIMS)
            case = {"kind": kind, "tokens": _log_int(rng, 200, 16384), "d": d, "h": h, "autocast": rng.random() < 0.4,
                    "outliers": rng.random() < 0.3}
        elif kind == "attn_train":
            case = {"kind": kind, "tokens": _log_int(rng, 200, 16384), "d": rng.choice(_ATTN_DIMS), "recipe": rng.choice(_RECIPES)}
        else:
            d, h, experts, top_k = rng.choice(_MOE_DIMS)
            lo, hi = (200, 16384) if kind == "moe_train" else (1, 4096)
            case = {"kind": kind, "tokens": _log_int(rng, lo, hi), "d": d, "h": h, "experts": experts, "top_k": top_k}
        if work(case)["flops"] <= _MOST_FLOPS:
            return case


# ---- inputs ----------------------------------------------------------------------------------------------------


def _randn(g, *shape, std=1.0, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=g, device="cuda").mul_(std).to(dtype)


def _fill(module, g):
    """Weights ~ N(0, 0.02), as trained projections have them."""
    with torch.no_grad():
        for p in module.parameters():
            p.copy_(torch.randn(p.shape, generator=g, device="cuda").mul_(0.02))
    return module


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind, tokens, d = case["kind"], case["tokens"], case["d"]
    state = {"kind": kind}
    if kind in ("mlp_fwd", "mlp_train"):
        autocast = case.get("autocast", False)
        model = FeedForward(d_model=d, hidden_size=case["h"], bias=False, dtype=torch.float32 if autocast else torch.bfloat16,
                            init_device="cuda")
        if kind == "mlp_fwd":
            Float8Config(ao=AOFloat8LinearConfig.recommended()).apply_float8_linear(model)
        else:
            Float8Config(ao_recipe=AOFloat8LinearRecipe.tensorwise).apply_float8_linear(model)
        state.update(model=_fill(model, g), autocast=autocast)
        x = torch.randn(tokens, d, generator=g, device="cuda")
        if case.get("outliers"):  # 0.1 % of the entries x100
            x.mul_(torch.where(torch.rand(tokens, d, generator=g, device="cuda") < 1e-3, 100.0, 1.0))
        state["x"] = x.to(torch.bfloat16)
    elif kind == "linear_fwd":
        model = torch.nn.Sequential(torch.nn.Linear(d, case["n"], bias=False, dtype=torch.bfloat16, device="cuda"))
        Float8Config(ao_recipe=AOFloat8LinearRecipe[case["recipe"]]).apply_float8_linear(model)
        state.update(model=_fill(model, g), x=_randn(g, tokens, d))
    elif kind == "attn_train":
        model = torch.nn.ModuleDict({k: torch.nn.Linear(d, d, bias=False, dtype=torch.bfloat16, device="cuda")
                                     for k in ("w_q", "w_k", "w_v", "w_out")})
        Float8Config(ao_recipe=AOFloat8LinearRecipe[case["recipe"]]).apply_float8_linear(model)
        # the output projection reads what attention made of q, k and v: an input of its own
        state.update(model=_fill(model, g), x=_randn(g, tokens, d), x_out=_randn(g, tokens, d).requires_grad_(True))
    else:
        experts, top_k = case["experts"], case["top_k"]
        mlp = DroplessMoEMLP(d_model=d, hidden_size=case["h"], num_experts=experts, dtype=torch.bfloat16, init_device="cuda",
                             keep_float8_weights=kind == "moe_fwd")
        state.update(model=ParallelDroplessMLP(mlp=_fill(mlp, g), top_k=top_k), x=_randn(g, tokens, d))
        # what the router hands over: skewed popularity (Zipf s = 1.1), so that with many experts some get no token
        rank = torch.arange(1, experts + 1, device="cuda", dtype=torch.float32)
        logits = torch.randn(tokens, experts, generator=g, device="cuda") - 1.75 * 1.1 * torch.log(rank)
        weights, indices = logits.softmax(-1).topk(top_k, dim=-1)
        state.update(expert_indices=indices, batch_size=torch.bincount(indices.flatten(), minlength=experts),
                     expert_weights=weights.to(torch.bfloat16))
    if kind.endswith("_train"):
        state["x"].requires_grad_(True)
        state["grad"] = _randn(g, tokens, d, std=1e-3)
        if kind == "moe_train":
            state["expert_weights"].requires_grad_(True)
    return state


# ---- one pass --------------------------------------------------------------------------------------------------


def run(state):
    kind, model, x = state["kind"], state["model"], state["x"]
    if kind in ("mlp_fwd", "linear_fwd"):
        with torch.no_grad():
            return model(x)
    if kind == "moe_fwd":
        with torch.no_grad():
            return model(x, state["expert_weights"], state["expert_indices"], state["batch_size"])
    model.zero_grad(set_to_none=True)
    x.grad = None
    out = {}
    if kind == "mlp_train":
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=state["autocast"]):
            y = model(x)
        y.backward(state["grad"])
    elif kind == "attn_train":
        x_out = state["x_out"]
        x_out.grad = None
        ys = [*float8_projections(x, model["w_q"], model["w_k"], model["w_v"]), model["w_out"](x_out)]
        torch.autograd.backward(ys, [state["grad"]] * 4)
        y = [t.detach() for t in ys]
        out["x_out_grad"] = x_out.grad
    else:
        weights = state["expert_weights"]
        weights.grad = None
        y = model(x, weights, state["expert_indices"], state["batch_size"])
        y.backward(state["grad"])
        out["expert_weights_grad"] = weights.grad
    out.update(y=y if isinstance(y, list) else y.detach(), x_grad=x.grad)
    for name, p in model.named_parameters():
        out[name] = p.grad
    return out


# ---- what a pass cannot do without ---------------------------------------------------------------------------------


def work(case):
    kind, tokens, d = case["kind"], case["tokens"], case["d"]
    act = 2.0 * tokens * d  # a bfloat16 [tokens, d] tensor
    if kind == "mlp_fwd":  # kept float8 weights in, x in, y out
        return {"bytes": 3.0 * d * case["h"] + 2 * act, "flops": 6.0 * tokens * d * case["h"]}
    if kind == "linear_fwd":
        return {"bytes": 2.0 * d * case["n"] + act + 2.0 * tokens * case["n"], "flops": 2.0 * tokens * d * case["n"]}
    if kind == "mlp_train":  # weights in and their gradients out, x and grad in, y and grad_x out
        size = 4 if case["autocast"] else 2
        return {"bytes": 2.0 * size * 3 * d * case["h"] + 4 * act, "flops": 18.0 * tokens * d * case["h"]}
    if kind == "attn_train":  # x, x_out and their gradients, four outputs; the gradient is one tensor
        return {"bytes": 2.0 * 2 * 4 * d * d + 9 * act, "flops": 24.0 * tokens * d * d}
    experts, slots, per_expert = case["experts"], tokens * case["top_k"], 3.0 * d * case["h"]
    if kind == "moe_train":
        return {"bytes": 4.0 * experts * per_expert + 4 * act, "flops": 6.0 * slots * per_expert}
    used = experts * (1.0 - (1.0 - 1.0 / experts) ** slots)  # experts that have a token
    return {"bytes": used * per_expert + 2 * act, "flops": 2.0 * slots * per_expert}


def tolerance(case):
    # Measured against the same operands multiplied in two halves of K, the second half first, by another tile kernel.
    # A single product differs by a bfloat16 rounding here and there (rel 1.2e-5).  Where a result is quantised again,
    # some roundings move a value to the next float8 code (rel 2.5e-4; one element of a gradient by 0.15 of its size
    # where outliers set the scale).  Summing the grad_input terms of several projections before rounding instead of
    # after gives rel 3.2e-3.
    kind = case["kind"]
    if kind == "linear_fwd":
        return {"rel": 1e-4, "max": 0.03}
    if kind in ("mlp_fwd", "moe_fwd"):
        return {"rel": 1e-3, "max": 0.06}
    return {"rel": 1e-2, "max": 0.4 if kind == "mlp_train" else 0.12}
