"""The tables of recorded sequences (olmo_core_amd/float8/plan.py), on the CPU."""

import itertools
import random
import types

import pytest
import torch

from olmo_core_amd.float8 import plan


def test_sizes_that_come_back_outlive_sizes_that_do_not():
    """A full table drops what was not replayed since it was last full; where everything was, its older half."""
    table, most = {}, plan._MOST_PLANS
    entry = lambda: types.SimpleNamespace(used=False)  # noqa: E731
    hot = table["hot"] = entry()
    for i in range(5 * most):
        hot.used = True  # (as every replay of it says)
        plan._remember(table, i, entry())
        assert len(table) <= most and table["hot"] is hot and i in table
    for e in table.values():
        e.used = True
    while len(table) < most:
        plan._remember(table, object(), entry())
    for e in table.values():
        e.used = True
    keys = list(table)
    plan._remember(table, "new", entry())
    assert list(table) == [*keys[-(most // 2):], "new"]


@pytest.mark.parametrize("fail, reason, warned", [
    (lambda p: p.float(), "tensor.float", False), (lambda p: p.to(torch.int32), "a conversion", False),
    (lambda p: p.to(device="cpu", dtype=torch.bfloat16), "a conversion", False), (lambda p: p[::2], "an index", False),
    (lambda p: p.device.place((plan._MOST_BYTES + 1,), torch.uint8), "more than _MOST_BYTES", False),
    (lambda p: {}["slot"], "KeyError: 'slot'", True), (lambda p: plan.ops.gemm_fp8(p, p, p, p), "TypeError: gemm_fp8: operands must be float8", True)])
def test_what_cannot_be_recorded_says_why(monkeypatch, caplog, fail, reason, warned):
    """A sequence that does what placeholders cannot has no plan and the reason; any other error is reported as well."""
    monkeypatch.setattr(plan, "_plans", {})
    monkeypatch.setattr(plan, "_seen", {})
    monkeypatch.setattr(plan, "_plannable", lambda inputs: True)
    x = torch.zeros(16, 16, dtype=torch.bfloat16)

    def fn(p):
        fail(p)
        return [], None

    for _ in range(6):
        assert plan.call(fn, [x], ("a test",)) is None
    (entry,) = plan._plans.values()
    assert entry.reason.startswith(reason)
    assert [r.levelname for r in caplog.records] == ["WARNING"] * warned


def test_sizes_met_twice_are_not_recorded(monkeypatch):
    """Two layers of one size, sequence lengths that come once: no recording, which costs more than a replay saves."""
    monkeypatch.setattr(plan, "_plans", {})
    monkeypatch.setattr(plan, "_seen", {})
    monkeypatch.setattr(plan, "_plannable", lambda inputs: True)
    recorded = []
    for tokens in range(1, 9):
        for _ in range(2):
            plan.call(lambda p: recorded.append(tokens) or p.float(), [torch.zeros(tokens, 16)], ("a test",))
    assert not recorded and not plan._plans
    plan.call(lambda p: recorded.append(3) or p.float(), [torch.zeros(3, 16)], ("a test",))
    assert recorded == [3] and len(plan._plans) == 1


def test_inputs_on_two_gpus_have_no_plan(monkeypatch):
    """A recorded sequence has one stream and takes no look at devices: an input that lives on another GPU goes to the calls one by
    one, which refuse it where they quantise it, however often its sizes were met and also where the sizes have a plan."""
    monkeypatch.setattr(plan, "_plans", {})
    monkeypatch.setattr(plan, "_seen", {})
    monkeypatch.setattr(plan, "_plannable", lambda inputs: True)
    monkeypatch.setattr(plan, "Plan", lambda *a: types.SimpleNamespace(run=lambda inputs: ([], None), used=False))
    on = lambda index: types.SimpleNamespace(shape=(16, 16), dtype=torch.bfloat16, get_device=lambda: index,  # noqa: E731
                                             device=types.SimpleNamespace(index=index))
    for own in (0, 1):
        for _ in range(4):
            assert plan.call(None, [on(0), None, on(1)], ("a test",), own=own) is None
        assert not plan._plans
    for _ in range(2):
        assert plan.call(None, [on(0), None, on(0)], ("a test",)) is None
    assert plan.call(None, [on(0), None, on(0)], ("a test",)) is not None
    assert plan.call(None, [on(0), None, on(1)], ("a test",)) is None


def test_temporaries_share_bytes_only_in_different_calls():
    """Intervals of calls that overlap get bytes of their own, all within the buffer; what has no call in common is reused."""
    rng = random.Random(1)
    for _ in range(300):
        calls = rng.randint(1, 20)
        t = {i: (rng.choice((0, 1, 255, 256, 257, rng.randint(1, 1 << 20))), *sorted(rng.choices(range(calls), k=2))) for i in range(rng.randint(0, 25))}
        at, size = plan._pack(t)
        assert at.keys() == t.keys() and all(a >= 0 and a % plan._ALIGN == 0 and a + t[i][0] <= size for i, a in at.items())
        for (i, a), (j, b) in itertools.combinations(at.items(), 2):
            if t[i][1] <= t[j][2] and t[j][1] <= t[i][2]:
                assert a + t[i][0] <= b or b + t[j][0] <= a
        rounded = {i: -(-v[0] // plan._ALIGN) * plan._ALIGN for i, v in t.items()}
        most = max((sum(rounded[i] for i, v in t.items() if v[1] <= c <= v[2]) for c in range(calls)), default=0)
        assert most <= size <= sum(rounded.values())
    assert plan._pack({"a": (512, 0, 1), "b": (512, 2, 3), "c": (100, 1, 2)}) == ({"a": 0, "b": 0, "c": 512}, 768)
    assert plan._pack({}) == ({}, 0)
