"""The calls a user of the attention step makes, as timed cases.

A case is one attention geometry and one call of it: `prepare` makes the
buffers and the plan that a serving program holds, `run` makes the call (over
several layers' caches for the short decode steps, as one token does), `exact`
is the same result in 64 bits. Buffers hold bf16 bits in the engine's layouts:
q and out token-major, the caches head-major.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "herbert-jit-bf16_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "herbert-jit-bf16_amd"))

import hsdpa  # noqa: E402

EPS = 1e-6
ROPE_THETA = 1e7
SINK = 1.25


def _case(name, kind, heads, kv_heads, head_dim, rows, past, layers=1, form="chained", sink=False, outliers=False,
          capacity=0):
    c = dict(kind=kind, heads=heads, kv_heads=kv_heads, head_dim=head_dim, rows=rows, past=past, layers=layers,
             form=form, sink=sink, outliers=outliers, capacity=capacity or past + rows)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one token after a short prompt, one layer: the smallest call, where
        # launches and latency are all there is
        _case("decode_1k", "attention", 8, 2, 256, 1, 1023),
        # one token of a long chat, through the caches of 8 layers (512 MiB:
        # more than the memory-side cache holds, as in a whole model)
        _case("decode_32k", "attention", 16, 2, 256, 1, 32767, layers=8),
        # one token over a very long document, with the outlier key channels
        # and value rows that trained models have
        _case("decode_128k_outliers", "attention", 16, 2, 256, 1, 131071, layers=2, outliers=True),
        # the reference's online-softmax decode form, head_dim 128, a ragged length
        _case("decode_fused_8k", "attention", 32, 4, 128, 1, 8190, layers=8, form="fused"),
        # a serving loop: one captured graph per token, rows and past read on
        # the device, the cache only partly filled
        _case("frame_20k", "frame", 16, 2, 256, 1, 19999, layers=8, capacity=32768),
        # verification of 8 drafted tokens over a long cache
        _case("verify_8_after_32k", "attention", 16, 2, 256, 8, 32768, layers=4),
        # a short prompt into an empty cache
        _case("prefill_512", "attention", 16, 4, 256, 512, 0),
        # a large chunk of a long prompt: the largest call
        _case("prefill_4096_after_8192", "attention", 16, 2, 256, 4096, 8192),
        # one pass of the engine (it sends at most 256 rows) through a gated
        # layer's whole chain: norms, RoPE, append, attention, gate
        _case("layer_256_after_8k", "layer", 16, 2, 256, 256, 8192),
        # a ragged chunk at head_dim 128, whose scale is no power of two
        _case("prefill_d128_2000_after_4100", "attention", 32, 4, 128, 2000, 4100),
        # a prompt into a model with the softmax sink, head_dim 64
        _case("prefill_sink_d64_1500_after_700", "attention", 32, 8, 64, 1500, 700, sink=True),
        # a prompt at a head dimension that is no power of two
        _case("prefill_d96_1000_after_500", "attention", 32, 8, 96, 1000, 500),
    ]


# query heads on KV heads: what the benchmark and the tests use
_GROUPS = [(8, 2), (16, 2), (16, 4), (32, 4), (32, 8), (12, 4), (16, 16)]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges: a decode step, a few rows, a
    prefill chunk, a layer pass or a frame step."""
    sort = rng.choice(["decode", "decode", "few", "prefill", "prefill", "prefill", "layer", "frame"])
    heads, kv = rng.choice(_GROUPS)
    dim = rng.choice([64, 128, 256, 256])
    if sort == "decode":
        if rng.random() < 0.25:
            dim = rng.choice([32, 96, 160, 192, 320, 512])
        n = _log_int(rng, 200, min(131072, 131072 * 512 // (kv * dim)))
        sink = rng.random() < 0.2
        return _case(None, "attention", heads, kv, dim, 1, n, layers=2, sink=sink, outliers=rng.random() < 0.2,
                     form="fused" if not sink and rng.random() < 0.3 else "chained")
    if sort == "few":
        return _case(None, "attention", heads, kv, dim, rng.randint(2, 16), _log_int(rng, 200, 40000))
    if sort == "frame":
        past = _log_int(rng, 100, 30000)
        return _case(None, "frame", heads, kv, dim, 1, past, layers=2, capacity=past + _log_int(rng, 64, 20000))
    if sort == "layer":
        return _case(None, "layer", heads, kv, dim, rng.choice([1, _log_int(rng, 2, 256), 256]),
                     _log_int(rng, 100, 16000))
    if rng.random() < 0.25:
        dim = rng.choice([32, 96, 160, 192, 320])
    rows = _log_int(rng, 17, 4096)
    past = rng.choice([0, _log_int(rng, 30, 12000)])
    limit = 4 * 16 * 256 * (4096 * 8192 + 4096 * 4097 // 2)          # the largest listed call
    if dim not in (64, 128, 256):
        limit //= 8                                                  # such models are smaller ones
    while 4 * heads * dim * (rows * past + rows * (rows + 1) // 2) > limit:
        rows, past = (rows + 1) // 2, past // 2
    return _case(None, "attention", heads, kv, dim, rows, past, sink=rng.random() < 0.2)


def _rotary(case):
    """The rotated dimensions of a gated layer's heads: a quarter, at least 32."""
    return max(32, case["head_dim"] // 4)


def _inputs(case, seed):
    """The case's tensors as bf16, on the GPU: N(0,1) q, K and V; a layer's
    projections before their norms, its weights and RoPE tables."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    rand = lambda *shape: torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)
    H, KV, D, R, cap = case["heads"], case["kv_heads"], case["head_dim"], case["rows"], case["capacity"]
    filled = case["past"] + R
    layers = []
    for _ in range(case["layers"]):
        k = torch.zeros(KV, cap, D, dtype=torch.bfloat16, device="cuda")
        v = torch.zeros_like(k)
        kf, vf = rand(KV, filled, D), rand(KV, filled, D)
        if case["outliers"]:
            ch = torch.randperm(D, generator=g, device="cuda")[:4]
            kf[:, :, ch] *= 20.0
            vf[:, torch.randperm(filled, generator=g, device="cuda")[:(filled + 99) // 100]] *= 8.0
        k[:, :filled], v[:, :filled] = kf, vf
        layers.append(dict(q=rand(R, H, D).bfloat16(), k=k, v=v))
    inp = dict(layers=layers)
    if case["kind"] == "layer":
        # q rows are [Q ; gate]
        inp["qg"] = (2.0 * rand(R, 2 * H * D)).bfloat16()
        inp["kp"] = (2.0 * rand(R, KV * D)).bfloat16()
        inp["vp"] = rand(R, KV * D).bfloat16()
        inp["q_norm"], inp["k_norm"] = (0.1 * rand(D)).bfloat16(), (0.1 * rand(D)).bfloat16()
        half = _rotary(case) // 2
        pos = torch.arange(cap, device="cuda", dtype=torch.float64)[:, None]
        ang = pos * ROPE_THETA ** (-torch.arange(half, device="cuda", dtype=torch.float64) / half)[None, :]
        inp["cos"], inp["sin"] = ang.cos().bfloat16(), ang.sin().bfloat16()
    return inp


def _scale(case):
    return float(np.float32(1.0 / math.sqrt(case["head_dim"])))


def prepare(case, seed):
    """The plan, its workspace and the buffers of every layer."""
    inp = _inputs(case, seed)
    H, KV, D, R = case["heads"], case["kv_heads"], case["head_dim"], case["rows"]
    kw = dict(form=case["form"], sink=case["sink"], max_rows=R)
    if case["kind"] == "layer":
        kw["q_row"] = 2 * H * D
    plan = hsdpa.Plan(H, H // KV, D, case["capacity"], **kw)
    st = dict(case=case, plan=plan, scale=_scale(case),
              ws=torch.empty(plan.workspace_bytes, dtype=torch.uint8, device="cuda"), **inp)
    st["outs"] = [torch.empty(R, H, D, dtype=torch.bfloat16, device="cuda") for _ in inp["layers"]]
    if case["kind"] == "layer":
        st["proj"] = torch.cat([inp["qg"].reshape(-1), inp["kp"].reshape(-1)])
        st["work"] = torch.empty_like(st["proj"])
        st["q"], st["kb"] = st["work"][:R * 2 * H * D], st["work"][R * 2 * H * D:]
    if case["kind"] == "frame":
        st["rows_dev"] = torch.tensor([1], dtype=torch.int64, device="cuda")
        st["past_dev"] = torch.tensor([case["past"]], dtype=torch.int64, device="cuda")
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        st["graph"], st["stream"] = torch.cuda.CUDAGraph(), stream

        def token():
            for l, out in zip(st["layers"], st["outs"]):
                plan.attention_frame_raw(l["q"].data_ptr(), l["k"].data_ptr(), l["v"].data_ptr(), out.data_ptr(),
                                         st["rows_dev"].data_ptr(), st["past_dev"].data_ptr(), st["scale"],
                                         st["ws"].data_ptr(), st["ws"].numel(), 0, stream.cuda_stream)

        with torch.cuda.stream(stream):
            token()
        torch.cuda.synchronize()
        with torch.cuda.graph(st["graph"], stream=stream):
            token()
    return st


def run(st):
    case = st["case"]
    if case["kind"] == "frame":
        st["graph"].replay()
        return st["outs"]
    if case["kind"] == "layer":
        H, KV, D = case["heads"], case["kv_heads"], case["head_dim"]
        l = st["layers"][0]
        # the projections land in the buffers that the chain updates in place
        st["work"].copy_(st["proj"])
        hsdpa.attention_layer_torch(st["plan"], st["q"], st["kb"], st["vp"], l["k"], l["v"], st["outs"][0],
                                    st["q_norm"], st["k_norm"], st["cos"], st["sin"], case["rows"], case["past"],
                                    st["scale"], EPS, st["ws"], KV * D, _rotary(case), gate=st["q"][H * D:],
                                    gate_row=2 * H * D, positions=case["capacity"])
        return [st["outs"][0], st["q"], st["kb"], l["k"], l["v"]]
    for l, out in zip(st["layers"], st["outs"]):
        hsdpa.attention_torch(st["plan"], l["q"], l["k"], l["v"], out, case["rows"], case["past"], st["scale"],
                              st["ws"], sink=SINK if case["sink"] else 0.0)
    return st["outs"]


def work(case):
    """K and V of the visible keys, q and the output once; two products over
    the visible (row, key) pairs. A layer's chain also reads and writes its
    projections, the appended rows and the gate once."""
    H, KV, D, R, P = case["heads"], case["kv_heads"], case["head_dim"], case["rows"], case["past"]
    nbytes = 2 * KV * (P + R) * D * 2 + 2 * R * H * D * 2
    if case["kind"] == "layer":
        nbytes += 2 * R * (H + KV) * D + 2 * R * H * D + 2 * 2 * R * KV * D
    return {"bytes": case["layers"] * nbytes, "flops": case["layers"] * 4 * H * D * (R * P + R * (R + 1) // 2)}


def tolerance(case):
    """The outputs are bf16: each is off by up to half a unit in its last
    place, 1.7e-3 of the result in the 2-norm (measured against `exact`:
    1.6e-3 to 1.7e-3 for the attention, 2.3e-3 for the layer's chain, whose
    output is rounded before and after the gate; the exponential's 6e-5 lies
    far below)."""
    return {"rel": 7e-3, "max": 0.02}


def _exact_attention(case, q, k, v):
    """softmax(scale q K^T) V in float64, causal after `past`, with the sink."""
    H, KV, D, R, P = case["heads"], case["kv_heads"], case["head_dim"], case["rows"], case["past"]
    g, n = H // KV, P + R
    out = torch.empty(R, H, D, dtype=torch.float64, device="cuda")
    step = max(1, (1 << 27) // (g * n))
    for y in range(KV):
        kt, vd = k[y, :n].double().t().contiguous(), v[y, :n].double()
        for r0 in range(0, R, step):
            r1 = min(R, r0 + step)
            s = torch.mm(q[r0:r1, y * g:(y + 1) * g].reshape(-1, D).double(), kt).mul_(_scale(case))
            s = s.view(r1 - r0, g, n)
            if R > 1:
                s.masked_fill_((torch.arange(n, device="cuda")[None, :]
                                > P + torch.arange(r0, r1, device="cuda")[:, None])[:, None, :], -math.inf)
            m = s.amax(dim=2, keepdim=True)
            if case["sink"]:
                m = m.clamp_min(SINK)
            e = s.sub_(m).exp_()
            den = e.sum(dim=2, keepdim=True)
            if case["sink"]:
                den = den + (SINK - m).exp()
            out[r0:r1, y * g:(y + 1) * g] = (torch.mm(e.view(-1, n), vd).view(r1 - r0, g, D)) / den
    return out


def _exact_norm_rope(case, x, w, cos, sin):
    """x * (1 + w) / rms(x), rounded to bf16 as the node stores it between the
    norm and the rotation, then the rotation of the leading dimensions."""
    R, half = case["rows"], _rotary(case) // 2
    x = x.double()
    y = x / (x.pow(2).mean(dim=-1, keepdim=True) + EPS).sqrt() * (1.0 + w.double())
    y = y.bfloat16().double()
    c = cos[case["past"]:case["past"] + R].double()[:, None, :]
    s = sin[case["past"]:case["past"] + R].double()[:, None, :]
    a, b = y[..., :half].clone(), y[..., half:2 * half].clone()
    y[..., :half], y[..., half:2 * half] = a * c - b * s, b * c + a * s
    return y


def exact(case, seed):
    inp = _inputs(case, seed)
    if case["kind"] != "layer":
        return [_exact_attention(case, l["q"], l["k"], l["v"]) for l in inp["layers"]]
    H, KV, D, R, P = case["heads"], case["kv_heads"], case["head_dim"], case["rows"], case["past"]
    k, v = inp["layers"][0]["k"], inp["layers"][0]["v"]
    qg = inp["qg"].double().clone()
    q = _exact_norm_rope(case, inp["qg"][:, :H * D].reshape(R, H, D), inp["q_norm"], inp["cos"], inp["sin"])
    qg[:, :H * D] = q.reshape(R, H * D)
    kn = _exact_norm_rope(case, inp["kp"].reshape(R, KV, D), inp["k_norm"], inp["cos"], inp["sin"])
    # the attention reads the bf16 buffers that the chain leaves
    k[:, P:P + R] = kn.bfloat16().transpose(0, 1)
    v[:, P:P + R] = inp["vp"].reshape(R, KV, D).transpose(0, 1)
    att = _exact_attention(case, q.bfloat16(), k, v)
    kd = k.double()
    kd[:, P:P + R] = kn.transpose(0, 1)
    gate = inp["qg"][:, H * D:].double().reshape(R, H, D)
    return [att / (1.0 + (-gate).exp()), qg.reshape(-1), kn.reshape(-1), kd, v.double()]
