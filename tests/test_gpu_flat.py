"""GPU parity of the causal prefill in equal shares (head_dim 128): row groups
walked by one, two and several workgroups, several row groups in one share, a
partial last row group and tile, 1 to 8 query heads per workgroup, the sink; the
output gate, padded rows and a captured graph on the same kernels."""
import numpy as np
import pytest
import torch

import hsdpa
import oracle
from hsdpa import workloads as W
from parity import assert_parity

from gpu_util import cus, run_hsdpa
from test_gpu_layer import Chain, run_fused, run_nodes
from test_gpu_strides import test_padded_strides as padded_strides

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


def _in_shares(plan, rows, past):
    return cus() != 256 or plan.route(rows, past)["splits"] == 0


def test_flat_gate(torch_cuda):
    """The gate in the epilogue and in the combine: bit for bit the gate node's."""
    c = Chain(24, 12, 128, 1333, 7, 1400, True, 64, seed=12)
    assert _in_shares(c.plan(), c.rows, c.past)
    fused, nodes = run_fused(torch_cuda, c), run_nodes(torch_cuda, c)
    for n in ("q", "k", "keys", "values", "out"):
        assert np.array_equal(fused[n], nodes[n]), n


def test_flat_padded_strides(torch_cuda):
    case = ("prefill_d128_shares", 16, 4, 128, 1812, 453)
    assert _in_shares(hsdpa.Plan(16, 4, 128, 1812 + 453), 1812, 453)
    padded_strides(torch_cuda, case)


def test_flat_graph_replays(torch_cuda):
    """A captured call, replayed with another call on the same workspace in
    between: every replay equals the eager result."""
    w = W.make("graph_shares", heads=32, kv_heads=8, head_dim=128, rows=1300, past=0, seed=44, capacity=3000)
    other = W.make("graph_other", heads=32, kv_heads=8, head_dim=128, rows=300, past=2500, seed=45, capacity=3000)
    plan = hsdpa.Plan(32, 4, 128, 3000)
    assert _in_shares(plan, w.rows, w.past)
    ws = torch.empty(plan.workspace_bytes, dtype=torch.uint8, device="cuda")
    dev = lambda x: [torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).cuda() for a in (x.q, x.k, x.v)]
    out = lambda x: torch.empty((x.rows, x.heads, x.head_dim), dtype=torch.int16, device="cuda")
    a, b, oa, ob = dev(w), dev(other), out(w), out(other)
    call = lambda x, t, o: hsdpa.attention_torch(plan, *t, o, x.rows, x.past, x.scale, ws)
    call(w, a, oa)
    torch.cuda.synchronize()
    eager = oa.clone()
    st = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        call(w, a, oa)
    for i in range(4):
        oa.fill_(-1)
        call(other, b, ob)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(oa, eager), i
