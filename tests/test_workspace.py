"""Plans that hsdpa_attention_static takes (their workspace within the static
scratch) keep fitting it: where the partials of pass 2 over all groups, or of
the causal prefill in equal shares, would not, the plan is laid out without
them."""
import pytest

import hsdpa

STATIC_SCRATCH = 32 << 20       # HSDPA_STATIC_SCRATCH_BYTES


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
