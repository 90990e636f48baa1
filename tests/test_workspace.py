"""Plans that hsdpa_attention_static takes (their workspace within the static
scratch) keep fitting it: where the partials of pass 2 over all groups, or of
the causal prefill in equal shares, would not, the plan is laid out without
them."""
import pytest

import hsdpa

STATIC_SCRATCH = 32 << 20       # HSDPA_STATIC_SCRATCH_BYTES


# MiB of a plan at head_dim 128 whose calls all have too few tiles for the equal
# shares, and of one whose longest call takes them
@pytest.mark.parametrize("heads,gqa,cap,rows,mib", [
    (8, 4, 1500, 0, 36),        # 1 144 tiles at most, of 2 048
    (8, 8, 1900, 0, 36),        # 1 830
    (4, 4, 6000, 100, 38),      # 100 rows at most
    (8, 4, 4060, 0, 71),
])
def test_shares_workspace(heads, gqa, cap, rows, mib):
    plan = hsdpa.Plan(heads, gqa, 128, cap, **({"max_rows": rows} if rows else {}))
    assert mib - 4 <= plan.workspace_bytes >> 20 <= mib
    taken = any(plan.route(r, cap - r)["splits"] == 0 for r in range(17, (rows or cap) + 1, 7))
    assert taken == (mib > 64)


@pytest.mark.parametrize("heads,gqa,dim,cap,rows", [
    (32, 8, 128, 30000, 8),     # four groups of columns, one round of pass-2 workgroups: 33 MiB otherwise
    (16, 8, 256, 12000, 16),    # eight groups
    (16, 8, 64, 8192, 0),       # any number of rows: the causal prefill's partials
    (32, 8, 96, 4096, 0),
])
def test_static_plans_fit(heads, gqa, dim, cap, rows):
    plan = hsdpa.Plan(heads, gqa, dim, cap, **({"max_rows": rows} if rows else {}))
    assert plan.workspace_bytes <= STATIC_SCRATCH
    n = min(rows or 500, 16)
    assert plan.route(n, cap - n)["main"] in ("few_rows", "causal_split", "causal")
