"""Activation checkpointing over converted modules (the reference wraps transformer blocks in
torch.utils.checkpoint: full / selected-blocks modes re-run the block's forward in backward, the selected-ops mode
saves only aten.mm / abs / max outputs, src/olmo_core/nn/utils.py:12-48, so the float8 operators are recomputed).
The re-run must reproduce the first run bit for bit: outputs and every gradient equal those of the plain call."""

from collections import defaultdict

import pytest
import torch
from torch.utils.checkpoint import CheckpointPolicy, checkpoint, create_selective_checkpoint_contexts

from helpers import seeded

pytestmark = pytest.mark.gpu

from olmo_core_amd.float8 import AOFloat8LinearRecipe, Float8Config, plan  # noqa: E402
from olmo_core_amd.float8.linear import float8_projections  # noqa: E402
from olmo_core_amd.nn import FeedForward  # noqa: E402


def _block(dev, recipe, fuse, D=512, H=1280):
    g = torch.Generator().manual_seed(5)
    ff = FeedForward(d_model=D, hidden_size=H, bias=False, dtype=torch.bfloat16, fuse_float8=fuse)
    with torch.no_grad():
        for p in ff.parameters():
            p.copy_((torch.randn(p.shape, generator=g) * 0.02).bfloat16())
    ff = ff.to(dev)
    Float8Config(ao_recipe=AOFloat8LinearRecipe(recipe)).apply_float8_linear(ff)
    return ff


def _selected_ops_context_fn():
    """The reference's policy: save mm (every second one) / abs / max, recompute the rest."""
    meta = defaultdict(int)
    save = {torch.ops.aten.mm.default, torch.ops.aten.abs.default, torch.ops.aten.max.default}

    def policy(ctx, func, *args, **kwargs):
        mode = "recompute" if ctx.is_recompute else "forward"
        if func == torch.ops.aten.mm.default:
            meta[f"{mode}_mm_count"] += 1
        to_save = func in save and not (func == torch.ops.aten.mm.default and meta[f"{mode}_mm_count"] % 2 == 0)
        return CheckpointPolicy.MUST_SAVE if to_save else CheckpointPolicy.PREFER_RECOMPUTE

    return create_selective_checkpoint_contexts(policy)


def _run(ff, x, go, wrap):
    for p in ff.parameters():
        p.grad = None
    xd = x.clone().requires_grad_(True)
    y = wrap(ff, xd)
    y.backward(go)
    return [y.detach().clone(), xd.grad.clone()] + [p.grad.clone() for p in ff.parameters()]


@pytest.mark.parametrize("recipe", ["tensorwise", "rowwise"])
@pytest.mark.parametrize("fuse", [True, False], ids=["fused", "per-linear"])
def test_checkpointed_block_reruns_bit_identically(dev, recipe, fuse):
    ff = _block(dev, recipe, fuse)
    x = seeded((3, 200, 512), 1).to(dev)  # (batch, seq, d_model)
    go = seeded((3, 200, 512), 2, std=1e-3).to(dev)
    plain = _run(ff, x, go, lambda m, t: m(t))
    full = _run(ff, x, go, lambda m, t: checkpoint(m, t, use_reentrant=False))
    selected = _run(ff, x, go, lambda m, t: checkpoint(m, t, use_reentrant=False, context_fn=_selected_ops_context_fn))
    names = ["y", "grad_x"] + [n for n, _ in ff.named_parameters()]
    for name, a, b, c in zip(names, plain, full, selected):
        assert torch.equal(a, b), f"{name}: full re-run differs from the plain call"
        assert torch.equal(a, c), f"{name}: selected-ops re-run differs from the plain call"


@pytest.mark.parametrize("recipe", ["tensorwise", "rowwise"])
@pytest.mark.parametrize("what", ["linear", "projections", "block"])
def test_sizes_whose_first_call_is_checkpointed(dev, monkeypatch, recipe, what):
    """No call on these sizes came before: the first run, its re-run in the backward, the same layer again and a second layer
    of its sizes save the same tensors, however often the sizes were met, and give the bits of plain calls."""
    monkeypatch.setattr(plan, "_plans", {})
    monkeypatch.setattr(plan, "_seen", {})
    if what == "block":
        layers = [_block(dev, recipe, True, 256, 512) for _ in range(2)]
    else:
        layers = [torch.nn.ModuleList([torch.nn.Linear(256, 256, bias=False, dtype=torch.bfloat16, device=dev) for _ in range(3)]) for _ in range(2)]
        for m in layers:
            Float8Config(ao_recipe=AOFloat8LinearRecipe(recipe)).apply_float8_linear(m)
    model = torch.nn.ModuleList(layers)
    one = {"block": lambda m, t: m(t), "linear": lambda m, t: m[0](t), "projections": lambda m, t: sum(float8_projections(t, *m))}[what]
    x, go = seeded((77, 256), 1).to(dev), seeded((77, 256), 2, std=1e-3).to(dev)

    def run(call):
        model.zero_grad()
        xd = x.clone().requires_grad_(True)
        y = xd
        for m in layers:
            y = call(lambda t, m=m: one(m, t), y)
        y.backward(go)
        return [y.detach(), xd.grad, *(p.grad for p in model.parameters() if p.grad is not None)]

    rerun = [run(lambda f, t: checkpoint(f, t, use_reentrant=False)) for _ in range(3)]
    plain = [run(lambda f, t: f(t)) for _ in range(3)]
    assert plan._plans  # (the plain calls' sizes have come back by now)
    rerun.append(run(lambda f, t: checkpoint(f, t, use_reentrant=False)))
    for got in (*plain[1:], *rerun):
        assert len(got) == len(plain[0]) and all(torch.equal(a, b) for a, b in zip(got, plain[0]))


def test_saved_tensor_hooks_see_the_tensors(dev, monkeypatch):
    """Hooks on saved tensors see the same ones on the first call of a set of sizes and on later ones."""
    monkeypatch.setattr(plan, "_plans", {})
    monkeypatch.setattr(plan, "_seen", {})
    ff = _block(dev, "tensorwise", True, 256, 512)
    seen = []
    for _ in range(4):
        packed = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append((t.shape, t.dtype)) or t, lambda t: t):
            ff(seeded((90, 256), 1).to(dev).requires_grad_(True)).sum().backward()
        seen.append(packed)
    assert len(seen[0]) == 13 and all(p == seen[0] for p in seen)
