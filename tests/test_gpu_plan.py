"""Recorded sequences of launches (olmo_core_amd/float8/plan.py): a layer's third call on one set of sizes, which records its
plan and replays it, has the bits of the first, which made its calls one by one."""

import pytest
import torch
import torch.nn as nn

from helpers import seeded
from olmo_core_amd.float8 import AOFloat8LinearConfig, AOFloat8LinearRecipe, Float8Config, plan
from olmo_core_amd.float8.linear import float8_projections
from olmo_core_amd.nn import DroplessMoEMLP, FeedForward, ParallelDroplessMLP

pytestmark = pytest.mark.gpu


@pytest.fixture
def runs(monkeypatch):
    """Plans replayed so far."""
    counted = []
    run = plan.Plan.run
    monkeypatch.setattr(plan, "_plans", {})
    monkeypatch.setattr(plan, "_seen", {})
    monkeypatch.setattr(plan.Plan, "run", lambda self, inputs: counted.append(1) or run(self, inputs))
    return counted


def _fill(m):
    with torch.no_grad():
        for i, p in enumerate(m.parameters()):
            p.copy_(seeded(tuple(p.shape), 11 + i, std=0.02))
    return m


def _step(model, x, fwd, gos, autocast=False):
    x = x.clone().requires_grad_(True)
    for p in model.parameters():
        p.grad = None
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
        ys = fwd(x)
    torch.autograd.backward(ys, gos)
    return [*(y.detach() for y in ys), x.grad, *(p.grad for p in model.parameters())]


def _check(step, runs, replays):
    """step(seed) -> tensors; other values between the calls that are compared."""
    want = {s: step(s) for s in (1,)}
    step(2)
    n = len(runs)
    want[2] = step(2)
    assert len(runs) - n == replays
    for s in (1, 2):
        for a, b in zip(step(s), want[s]):
            assert (a is None) == (b is None) and (a is None or (a.dtype == b.dtype and torch.equal(a, b)))


@pytest.mark.parametrize("tokens, d, h", [(1, 256, 512), (40, 1040, 272), (300, 256, 512), (1999, 512, 1408), (2000, 2048, 8192)])
@pytest.mark.parametrize("autocast", [False, True])
def test_feed_forward(dev, runs, tokens, d, h, autocast):
    model = FeedForward(d_model=d, hidden_size=h, bias=False, dtype=torch.float32 if autocast else torch.bfloat16, init_device="cuda")
    Float8Config(ao_recipe=AOFloat8LinearRecipe.tensorwise).apply_float8_linear(_fill(model))
    go = seeded((d, tokens), 5, std=1e-3).to(dev).t()  # (not contiguous)
    _check(lambda s: _step(model, seeded((tokens, d), s).to(dev), lambda x: [model(x)], [go], autocast), runs, 2)


def test_replays_hold_no_more_than_the_calls(dev, runs):
    """A block whose backward, call by call, gives back half of its temporaries before it takes the next: so does its plan."""
    model = FeedForward(d_model=1024, hidden_size=2816, bias=False, dtype=torch.bfloat16, init_device="cuda")
    Float8Config(ao_recipe=AOFloat8LinearRecipe.tensorwise).apply_float8_linear(_fill(model))
    go, peaks = seeded((12000, 1024), 5, std=1e-3).to(dev), []

    def step(s):
        x = seeded((12000, 1024), s).to(dev)
        torch.cuda.reset_peak_memory_stats()
        held = torch.cuda.memory_allocated()
        out = _step(model, x, lambda t: [model(t)], [go])
        peaks.append(torch.cuda.max_memory_allocated() - held)
        return out

    _check(step, runs, 2)
    assert peaks[-1] <= 1.05 * peaks[0]


@pytest.mark.parametrize("tokens", [1, 16, 23, 65, 777])
def test_evaluation(dev, runs, tokens):
    model = FeedForward(d_model=256, hidden_size=768, bias=False, dtype=torch.bfloat16, init_device="cuda")
    Float8Config(ao=AOFloat8LinearConfig.recommended()).apply_float8_linear(_fill(model))
    with torch.no_grad():
        _check(lambda s: [model(seeded((tokens, 256), s).to(dev))], runs, 1)
        model.w2.weight.mul_(-1.0)  # kept float8 weights are made again
        a = model(seeded((tokens, 256), 1).to(dev))
        model.w2.weight.mul_(-1.0)
        assert torch.equal(a, -model(seeded((tokens, 256), 1).to(dev)))


@pytest.mark.parametrize("recipe", ["tensorwise", "rowwise", "rowwise_with_gw_hp"])
@pytest.mark.parametrize("tokens", [7, 333])
def test_projections(dev, runs, recipe, tokens):
    model = nn.ModuleDict({k: nn.Linear(256, n, bias=False, dtype=torch.bfloat16, device=dev) for k, n in (("q", 256), ("k", 128), ("v", 128), ("o", 320))})
    Float8Config(ao_recipe=AOFloat8LinearRecipe[recipe]).apply_float8_linear(_fill(model))
    model["k"].weight.requires_grad_(False)
    gos = [seeded((tokens, n), 20 + i, std=1e-3).to(dev) for i, n in enumerate((256, 128, 128, 320))]
    fwd = lambda x: [*float8_projections(x, model["q"], model["k"], model["v"]), model["o"](x)]  # noqa: E731
    planned = 0 if recipe == "rowwise_with_gw_hp" else 4
    _check(lambda s: _step(model, seeded((tokens, 256), s).to(dev), fwd, gos), runs, planned)
    with torch.no_grad():
        _check(lambda s: [model["o"](seeded((tokens, 256), s).to(dev))], runs, 1)


def test_experts(dev, runs):
    mlp = DroplessMoEMLP(d_model=256, hidden_size=128, num_experts=8, dtype=torch.bfloat16, init_device="cuda", keep_float8_weights=True)
    layer = ParallelDroplessMLP(mlp=_fill(mlp), top_k=2)

    def step(s):
        g = torch.Generator(device=dev).manual_seed(s)
        weights, ids = torch.randn(48, 8, generator=g, device=dev).softmax(-1).topk(2, dim=-1)
        with torch.no_grad():
            return [layer(seeded((48, 256), s).to(dev), weights.bfloat16(), ids, torch.bincount(ids.flatten(), minlength=8))]

    _check(step, runs, 1)


def test_sizes_that_do_not_come_back_are_not_recorded(dev, runs):
    lin = nn.Sequential(nn.Linear(128, 128, bias=False, dtype=torch.bfloat16, device=dev))
    Float8Config(ao_recipe=AOFloat8LinearRecipe.tensorwise).apply_float8_linear(lin)
    with torch.no_grad():
        for tokens in range(1, 9):
            lin(seeded((tokens, 128), 1).to(dev))
    assert not plan._plans and len(plan._seen) == 8 and not runs


@pytest.mark.parametrize("name, tokens, kept", [
    ("swiglu_fwd", 300, False), ("few_rows_swiglu", 23, True), ("few_rows_cast_gemm", 3, True), ("gemm_fp8_swiglu", 4096, False),
    ("gemm_fp8_codes", 4096, False), ("swiglu_bwd_cast", 300, False), ("gemm_fp8_products", 300, False), ("cast_tensorwise", 300, False)])
def test_replaced_operations_are_called(dev, runs, monkeypatch, name, tokens, kept):
    """An operation that is replaced after its calls were recorded is called again."""
    model = FeedForward(d_model=256, hidden_size=2048, bias=False, dtype=torch.bfloat16, init_device="cuda")
    Float8Config(ao=AOFloat8LinearConfig.recommended() if kept else AOFloat8LinearConfig()).apply_float8_linear(_fill(model))
    x, go = seeded((tokens, 256), 1).to(dev), seeded((tokens, 256), 2, std=1e-3).to(dev)

    def step():
        if not kept:
            return _step(model, x, lambda t: [model(t)], [go])
        with torch.no_grad():
            return [model(x)]

    want = [step() for _ in range(4)][-1]
    n, called, real = len(runs), [], getattr(plan.ops, name)
    assert n
    monkeypatch.setattr(plan.ops, name, lambda *a, **k: called.append(1) or real(*a, **k))
    got = step()
    assert called and len(runs) == n and all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("kept, autocast", [(True, False), (False, True)])
def test_forms_without_a_plan_are_not_looked_up(dev, runs, kept, autocast):
    """Training with kept float8 weights, and float32 activations under autocast, have no plans: no lookup, no attempt."""
    model = nn.ModuleDict({"ff": FeedForward(d_model=256, hidden_size=512, bias=False, dtype=torch.bfloat16, init_device="cuda"),
                           "q": nn.Linear(256, 256, bias=False, dtype=torch.bfloat16, device=dev),
                           "k": nn.Linear(256, 256, bias=False, dtype=torch.bfloat16, device=dev)})
    Float8Config(ao=AOFloat8LinearConfig.recommended() if kept else AOFloat8LinearConfig()).apply_float8_linear(_fill(model))
    x = seeded((300, 256), 1).to(dev)
    x, go = (x.float() if autocast else x), seeded((300, 256), 2, std=1e-3).to(dev)
    fwd = lambda t: [model["ff"](t), *float8_projections(t, model["q"], model["k"])]  # noqa: E731
    got = [_step(model, x, fwd, [go] * 3, autocast) for _ in range(4)]
    assert not plan._seen and not plan._plans and not runs
    assert all(torch.equal(a, b) for a, b in zip(got[0], got[3]))
