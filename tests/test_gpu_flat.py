"""GPU parity of the causal prefill in equal shares (head_dim 128): row groups
walked by one, two and several workgroups, several row groups in one share, a
partial last row group and tile, 1 to 8 query heads per workgroup, the sink."""
import numpy as np
import pytest
import torch

import hsdpa
import oracle
from hsdpa import workloads as W
from parity import assert_parity

from gpu_util import cus, run_hsdpa

pytestmark = pytest.mark.gpu

CASES = [
    # name, heads, kv_heads, rows, past, sink
    ("g4_1300_rows_no_cache", 32, 8, 1300, 0, None),
    ("g2_partial_row_group", 24, 12, 1333, 7, None),
    ("g1_seven_tiles_over", 40, 40, 900, 513, None),
    ("g8_sink", 32, 4, 700, 905, 6.0),
    ("g8_sink_no_cache", 16, 2, 2050, 0, 5.0),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_flat_parity(torch_cuda, case):
    name, h, kvh, rows, past, sink = case
    w = W.make(name, heads=h, kv_heads=kvh, head_dim=128, rows=rows, past=past, seed=57)
    plan = hsdpa.Plan(w.heads, w.gqa, w.head_dim, w.capacity, sink=sink is not None)
    print(f"case {name} {plan.route(rows, past)}", flush=True)
    if cus() == 256:                # the shapes are chosen for 256 compute units
        assert plan.route(rows, past)["splits"] == 0, "not in equal shares"
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
