"""The tables of recorded sequences (olmo_core_amd/float8/plan.py), on the CPU."""

import types

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
