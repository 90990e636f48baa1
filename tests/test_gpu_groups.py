"""GPU parity of pass 2 over all the groups of a KV head per workgroup
(decode_pv_groups: head_dim 128 and 256, past one round of 256-key workgroups
per group), at the edges of its runs and chunks: 1 to 8 groups (its instantiations
hold 1, 2, 4 and 8), a group count below the instantiation's, padded columns,
runs of 4 tiles and of one tile more than a chunk, a partial last tile and a
last workgroup with less than the others, and the sink. 16 KV heads, so that a
run has one sixteenth of the tiles."""
import pytest

import hsdpa
import oracle
from hsdpa import workloads as W
from parity import assert_parity

from gpu_util import cus, run_hsdpa

pytestmark = pytest.mark.gpu

CASES = [
    # name, heads, kv_heads, rows, past, sink (head_dim 256)
    ("one_group_8_columns_9_tile_runs", 128, 16, 1, 4096, None),     # 129 tiles: one over 8 per run
    ("one_group_16_columns_partial_tile", 128, 16, 2, 4300, None),
    ("one_group_9_columns", 48, 16, 3, 8190, None),
    ("two_groups_5_tile_runs", 128, 16, 4, 2300, None),
    ("two_groups_12_tile_runs", 128, 16, 4, 6100, None),
    ("three_groups_of_four", 128, 16, 6, 1500, None),
    ("four_groups_one_key_past_a_tile", 128, 16, 8, 1273, None),     # 1281 keys
    ("four_groups_9_tile_runs", 16, 2, 8, 32768, None),
    ("five_groups_padded", 128, 16, 9, 900, None),                   # 72 columns: 5 groups of 15
    ("eight_groups", 128, 16, 16, 700, None),
    ("eight_groups_several_chunks", 16, 2, 16, 16500, None),
    ("one_row_32_heads_per_kv_head", 256, 8, 1, 5000, None),
    ("two_groups_sink", 128, 16, 4, 2300, 6.0),
    ("one_group_sink", 128, 16, 2, 4300, 8.0),
]


# head_dim 128: runs of 6 tiles or more, chunks of 8 tiles up to 4 groups, of 4 beyond
CASES_128 = [
    ("d128_one_group_9_tile_runs", 128, 16, 2, 4300, None),
    ("d128_two_groups_7_tile_runs", 128, 16, 4, 3100, None),
    ("d128_three_groups_of_four", 128, 16, 6, 3300, None),
    ("d128_four_groups_6_tile_runs", 128, 16, 8, 2900, None),
    ("d128_four_groups_two_chunks", 32, 4, 8, 20011, None),
    ("d128_eight_groups_6_tile_runs", 128, 16, 16, 2600, None),
    ("d128_two_groups_sink", 128, 16, 4, 3100, 6.0),
]
ALL = [c + (256,) for c in CASES] + [c + (128,) for c in CASES_128]


@pytest.mark.parametrize("case", ALL, ids=[c[0] for c in ALL])
def test_groups_parity(torch_cuda, case):
    name, h, kvh, rows, past, sink, dim = case
    import numpy as np
    import torch

    w = W.make(name, heads=h, kv_heads=kvh, head_dim=dim, rows=rows, past=past, seed=91)
    plan = hsdpa.Plan(w.heads, w.gqa, w.head_dim, w.capacity, sink=sink is not None)
    print(f"case {name}", flush=True)
    if cus() == 256:                # the shapes are chosen for 256 compute units
        assert plan.route(rows, past)["splits"] == 0, "not over all groups"
    if sink is None:
        out, ref = run_hsdpa(w, plan), oracle.attention(w)
    else:
        dev = [torch.from_numpy(np.ascontiguousarray(x).view(np.int16)).cuda() for x in (w.q, w.k, w.v)]
        o = torch.full((w.rows, w.heads, w.head_dim), -1, dtype=torch.int16, device="cuda")
        ws = torch.empty(plan.workspace_bytes, dtype=torch.uint8, device="cuda")
        hsdpa.attention_torch(plan, *dev, o, w.rows, w.past, w.scale, ws, sink=sink)
        torch.cuda.synchronize()
        out, ref = o.cpu().numpy().view(np.uint16), oracle.attention(w, sink=sink)
    assert_parity(out, ref, w, name)


# plans whose workspace holds fewer workgroups, at rows and lengths where that
# decides the form (name, heads, kv_heads, head_dim, rows, past, capacity, max_rows, over all groups)
SMALLER = [
    ("static_16_rows", 16, 2, 256, 16, 6000, 12000, 16, False),
    ("static_12_rows_full", 16, 2, 256, 12, 11988, 12000, 16, False),
    ("static_8_rows", 16, 2, 256, 8, 11900, 12000, 16, True),
    ("short_cache_11_rows", 128, 16, 256, 11, 610, 621, 11, True),
    ("static_d128_8_rows", 32, 4, 128, 8, 29000, 30000, 8, False),
]


@pytest.mark.parametrize("case", SMALLER, ids=[c[0] for c in SMALLER])
def test_smaller_workspaces(torch_cuda, case):
    name, h, kvh, dim, rows, past, cap, max_rows, groups = case
    w = W.make(name, heads=h, kv_heads=kvh, head_dim=dim, rows=rows, past=past, seed=92, capacity=cap)
    plan = hsdpa.Plan(w.heads, w.gqa, w.head_dim, cap, max_rows=max_rows)
    print(f"case {name} {plan.route(rows, past)}", flush=True)
    if cus() == 256:
        assert plan.workspace_bytes <= 32 << 20
        assert (plan.route(rows, past)["splits"] == 0) == groups
    assert_parity(run_hsdpa(w, plan), oracle.attention(w), w, name)
