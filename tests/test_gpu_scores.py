"""GPU parity of the exponentials over the whole range of scores, on every kernel
that takes them from the dot products in one step (the causal forms) or from
the scores over all groups: scores of about 1e6 whose differences are small
(with the sink beside the maximum), of 1e10 and 1e30, negative scales, and a
scale so small that the difference of two dot products leaves the f32 range.

The dot products are exact: one pair of elements gives every key 2^23, the
others small integers, all times one power of two, so that any order of
summation gives the same f32 and the weights of the oracle are known to the
last bit of its exponential; the parity criterion then holds as it stands."""
import numpy as np
import pytest
import torch

import hsdpa
import oracle
from hsdpa import workloads as W
from parity import assert_parity, bf16_f32

pytestmark = pytest.mark.gpu

CASES = [
    # name, heads, kv_heads, head_dim, rows, past, sink, kernels (None: not pinned here)
    ("causal_256", 16, 4, 256, 40, 0, False, "causal"),
    ("causal_96_sink", 4, 4, 96, 100, 40, True, "causal"),
    ("causal_320", 8, 8, 320, 200, 0, False, "causal"),
    ("short_64", 8, 2, 64, 40, 700, False, "causal_short"),
    ("short_256", 4, 1, 256, 64, 900, False, "causal_short"),
    ("split_64", 8, 2, 64, 300, 1500, False, "causal_split"),
    ("split_256_sink", 4, 1, 256, 64, 900, True, "causal_split"),
    ("paired_64", 16, 2, 64, 2200, 0, False, "causal_paired"),
    ("paired_64_sink", 16, 2, 64, 2200, 0, True, "causal_paired"),
    ("shares_128", 32, 8, 128, 1300, 0, False, None),
    ("shares_128_sink", 32, 4, 128, 700, 905, True, None),
    ("groups_256", 128, 16, 256, 4, 2300, False, "few_rows"),
    ("groups_256_sink", 128, 16, 256, 4, 2300, True, "few_rows"),
    ("groups_128", 128, 16, 128, 4, 3100, False, "few_rows"),
]
# the power of two on the dot products, and the scale
LEVELS = {"1e6": (0, 2.0 ** -3), "1e6_negative": (0, -(2.0 ** -3)), "1e10": (13, 2.0 ** -3), "1e30": (80, 2.0 ** -3)}


def _workload(name, h, kvh, d, rows, past, e, scale, signs=False):
    """Dot products of 2^e (+-2^23 + small integers); a negative scale makes
    the smallest of them the largest score."""
    n = past + rows
    ints = lambda seed, shape: (W.splitmix64(seed, int(np.prod(shape))) % np.uint64(7)).astype(np.float32).reshape(shape) - 3
    q, k = ints(5, (rows, h, d)), ints(6, (kvh, n, d))
    q[..., 0], k[..., 0] = 2.0 ** 12, 2.0 ** 11
    if signs:
        k[..., 0] *= np.where(W.splitmix64(8, kvh * n).reshape(kvh, n) & np.uint64(1), 1.0, -1.0)
    q, k = q * np.float32(2.0 ** (e // 2)), k * np.float32(2.0 ** (e - e // 2))
    return W.Workload(name, h, kvh, d, rows, past, n, W.f32_to_bf16(q), W.f32_to_bf16(k),
                      W.normal_bf16(7, (kvh, n, d)), float(np.float32(scale)))


def _run(w, sink=None):
    plan = hsdpa.Plan(w.heads, w.gqa, w.head_dim, w.capacity, sink=sink is not None)
    print(f"case {w.name} {plan.route(w.rows, w.past)}", flush=True)
    dev = [torch.from_numpy(np.ascontiguousarray(x).view(np.int16)).cuda() for x in (w.q, w.k, w.v)]
    out = torch.full((w.rows, w.heads, w.head_dim), -1, dtype=torch.int16, device="cuda")
    ws = torch.empty(plan.workspace_bytes, dtype=torch.uint8, device="cuda")
    hsdpa.attention_torch(plan, *dev, out, w.rows, w.past, w.scale, ws, sink=0.0 if sink is None else sink)
    torch.cuda.synchronize()
    return plan, out.cpu().numpy().view(np.uint16)


@pytest.mark.parametrize("level", LEVELS)
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_large_scores(torch_cuda, case, level):
    name, h, kvh, d, rows, past, sink, kernels = case
    e, scale = LEVELS[level]
    w = _workload(f"{name}_{level}", h, kvh, d, rows, past, e, scale)
    # beside the row maxima (the keys' standard deviation is 4 sqrt(D) in the
    # dot product): some lie above the sink, some below
    near = abs(scale) * 2.0 ** e * (2.0 ** 23 * np.sign(scale) + 12.5 * d ** 0.5)
    s = float(np.float32(near)) if sink else None
    plan, out = _run(w, s)
    if kernels:
        assert plan.route(rows, past)["main"] == kernels
    assert_parity(out, oracle.attention(w, sink=s), w, w.name)


@pytest.mark.parametrize("case", [c for c in CASES if not c[6]], ids=[c[0] for c in CASES if not c[6]])
def test_tiny_scale(torch_cuda, case):
    """Dot products of +-2^127: their differences leave the f32 range, the
    scores +-2."""
    name, h, kvh, d, rows, past, _, _ = case
    w = _workload(f"{name}_tiny", h, kvh, d, rows, past, 104, 2.0 ** -126, signs=True)
    _, out = _run(w)
    assert_parity(out, oracle.attention(w), w, w.name)


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_overflowing_scores(torch_cuda, case):
    """Scores past the f32 range: the largest is infinite, its difference from
    itself a NaN, which the exponential clamps like the others' -inf, so that every
    key weighs the same, 2^-126. Those weights' products are at the edge of what
    the matrix cores keep (smaller ones are flushed, an error of 1 a key at most before
    the division by the number of keys), so the outputs are not compared one by one: over
    32 keys or more the mean of N(0,1) values lies below 1 (6 of its deviations), the
    flushed products add 1 at most, and a single key's values, as one infinite score would give
    them, pass 2 in a row of 64 values or more almost surely."""
    name, h, kvh, d, rows, past, sink, _ = case
    w = W.make(name, heads=h, kv_heads=kvh, head_dim=d, rows=rows, past=past, seed=34, scale=3e38)
    s = 3.0 if sink else None
    _, out = _run(w, s)
    assert np.isfinite(bf16_f32(out)).all()
    for x in (out, oracle.attention(w, sink=s)):
        x = np.abs(bf16_f32(x).reshape(rows, h, d))[max(0, 31 - past):]
        assert x.max() <= 2.0


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_negative_scale(torch_cuda, case):
    name, h, kvh, d, rows, past, sink, _ = case
    w = W.make(name, heads=h, kv_heads=kvh, head_dim=d, rows=rows, past=past, seed=33, scale=-1.0 / d ** 0.5)
    s = 1.25 if sink else None
    _, out = _run(w, s)
    assert_parity(out, oracle.attention(w, sink=s), w, w.name)
