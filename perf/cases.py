"""The calls that this framework is used for, as cases that can be timed and compared.

Three kinds of call, each through a public entry point:

  block   MoEBlock.launch: router, permutation, experts and combine of one layer on normalised
          rows, with the routing results and the per-expert rows that the call hands back
  stack   MoEStack.launch: RMSNorm, block and residual of one or several layers, as a decoding
          or prefilling program drives them
  ops     the tensor operations of the C ABI, in the order in which an expert executor written
          against them runs one expert's MLP: gate and up products, SiLU, product, down product
          (INT8 weights: hm_matmul_w8a32, FP32 weights: hm_matmul_f32)

Weights are N(0, 0.02), INT8 ones packed per projection with scale max|w| / 127 and zero point 0;
hidden rows are N(0, 1), divided by their root mean square where a call expects normalised rows.
Everything is drawn on the GPU from the seed alone.
"""
from __future__ import annotations

import ctypes as C
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "hypermoe-engine_amd"))

from hmoe import capi  # noqa: E402
from hmoe.block import DeviceExpertLayer, MoEBlock  # noqa: E402
from hmoe.stack import MoEStack  # noqa: E402

_EPS = 1e-6
_BLOCK_OUT = ("out", "ids", "scores", "counts", "offsets", "perm_tokens", "perm_weights",
              "expert_out")


def _case(name, kind, dtype, tokens, hidden=2048, inter=768, experts=128, top_k=8, layers=1,
          skew=False):
    c = dict(kind=kind, dtype=dtype, tokens=tokens, hidden=hidden, inter=inter, experts=experts,
             top_k=top_k, layers=layers, skew=skew)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # one user's decode step through a few layers of the 128-expert top-8 stack: the smallest
        # call, bound by latency and launches
        _case("stack_int8_decode_1", "stack", "int8", 1, layers=4),
        # a decode batch of 16 sequences
        _case("block_int8_decode_16", "block", "int8", 16),
        # a decode batch off every tile and wave size, four rows an expert
        _case("block_int8_decode_61", "block", "int8", 61),
        # a chunk of a prompt, ragged, about twenty rows an expert
        _case("block_int8_chunk_333", "block", "int8", 333),
        # a 2048-token prefill of one layer with its norm and residual
        _case("stack_int8_prefill_2048", "stack", "int8", 2048),
        # the largest prefill, routing skewed as trained routers skew it (one expert has ten times
        # the mean load)
        _case("block_int8_prefill_4096", "block", "int8", 4096, skew=True),
        # a layer whose sizes are off the usual grid: 60 experts, an intermediate of 11 x 64, an
        # odd number of tokens
        _case("block_int8_offgrid_201", "block", "int8", 201, hidden=1024, inter=704, experts=60,
              top_k=4),
        # unquantised experts: a decode batch and a prefill
        _case("block_fp32_decode_16", "block", "fp32", 16, experts=64),
        _case("block_fp32_prefill_512", "block", "fp32", 512, experts=64),
        # one expert at a time through the tensor operations: a single row, and the rows that an
        # expert collects in a prefill
        _case("ops_int8_1", "ops", "int8", 1, experts=1, top_k=1),
        _case("ops_int8_300", "ops", "int8", 300, experts=1, top_k=1),
        _case("ops_fp32_150", "ops", "fp32", 150, experts=1, top_k=1),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["block_int8", "block_int8", "block_int8", "stack", "block_fp32", "offgrid",
                       "ops_int8", "ops_fp32"])
    if kind == "block_int8":
        return _case(None, "block", "int8", _log_int(rng, 1, 4000), skew=rng.random() < 0.5)
    if kind == "stack":
        t = _log_int(rng, 1, 2500)
        return _case(None, "stack", "int8", t, layers=rng.randint(1, 4) if t <= 4 else 1)
    if kind == "block_fp32":
        return _case(None, "block", "fp32", _log_int(rng, 1, 700), experts=rng.choice([8, 16, 64]))
    if kind == "offgrid":
        experts = rng.randint(8, 100)
        return _case(None, "block", "int8", _log_int(rng, 1, 600), hidden=64 * rng.randint(8, 32),
                     inter=16 * rng.randint(16, 64), experts=experts, top_k=rng.randint(1, 8),
                     skew=rng.random() < 0.5)
    odd = rng.random() < 0.25
    hidden = 64 * rng.randint(8, 48) + (rng.randint(1, 63) if odd else 0)
    inter = 32 * rng.randint(8, 48) + (rng.randint(1, 31) if odd else 0)
    return _case(None, "ops", "int8" if kind == "ops_int8" else "fp32", _log_int(rng, 1, 800),
                 hidden=hidden, inter=inter, experts=1, top_k=1)


# ---- inputs -----------------------------------------------------------------------------------

def _gen(seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + what)
    return g


def _weights(case, seed, layer):
    """([E, 3, H*I] payload gate | up | down, [E, 3] scales or None) on the GPU."""
    e, n = case["experts"], case["hidden"] * case["inter"]
    g = _gen(seed, 100 + layer)
    if case["dtype"] == "fp32":
        return torch.empty((e, 3, n), dtype=torch.float32, device="cuda").normal_(0, 0.02, generator=g), None
    q = torch.empty((e, 3, n), dtype=torch.int8, device="cuda")
    scale = torch.empty((e, 3), dtype=torch.float32, device="cuda")
    for i in range(0, e, 16):
        w = torch.empty((min(16, e - i), 3, n), dtype=torch.float32, device="cuda").normal_(0, 0.02, generator=g)
        s = w.abs().amax(dim=2) / 127.0
        scale[i:i + 16] = s
        q[i:i + 16] = torch.round(w / s[:, :, None]).clamp_(-127, 127).to(torch.int8)
    return q, scale


def _router(case, seed, layer):
    h, e = case["hidden"], case["experts"]
    w = torch.empty((h, e), dtype=torch.float32, device="cuda").normal_(0, 0.02, generator=_gen(seed, 200 + layer))
    if case["skew"]:  # the last feature is a constant 1: its router row is a bias, Zipf over the experts
        rank = torch.randperm(e, generator=_gen(seed, 300 + layer), device="cuda").float() + 1
        w[-1] = -0.9 * 1.1 * torch.log(rank)
    return w


def _rows(case, seed):
    x = torch.empty((case["tokens"], case["hidden"]), dtype=torch.float32, device="cuda").normal_(generator=_gen(seed, 1))
    if case["kind"] == "stack":
        return x  # the stack normalises
    x = x / torch.sqrt(x.square().mean(dim=1, keepdim=True) + _EPS)
    if case["skew"]:
        x[:, -1] = 1.0
    return x


def _layer(case, seed, layer):
    q, scale = _weights(case, seed, layer)
    payload = q.cpu().numpy()
    del q
    if case["dtype"] == "fp32":
        return DeviceExpertLayer(payload, None, None, case["hidden"], case["inter"])
    return DeviceExpertLayer(payload, scale.cpu().numpy(), np.zeros((case["experts"], 3), np.int32),
                             case["hidden"], case["inter"])


def _prepare_ops(case, seed):
    m, h, i = case["tokens"], case["hidden"], case["inter"]
    q, scale = _weights(case, seed, 0)
    f = dict(dtype=torch.float32, device="cuda")
    s = dict(kind="ops", x=_rows(case, seed), w=[q[0, p].clone() for p in range(3)],
             dims=[(h, i), (h, i), (i, h)], gate=torch.empty((m, i), **f), up=torch.empty((m, i), **f),
             act=torch.empty((m, i), **f), z=torch.empty((m, i), **f), y=torch.empty((m, h), **f))
    if case["dtype"] == "int8":
        s["scale"] = [float(v) for v in scale[0].cpu()]
        need = 1
        for k, n in s["dims"]:
            plan = capi.HmInt8GemmPlan()
            capi.call("hm_plan_int8_gemm", m, k, n, 0, C.byref(plan))
            need = max(need, plan.scratch_elements)
        s["scratch"] = torch.empty(need, **f)
    return s


def prepare(case, seed):
    if case["kind"] == "ops":
        return _prepare_ops(case, seed)
    layers = [_layer(case, seed, n) for n in range(case["layers"])]
    routers = [_router(case, seed, n) for n in range(case["layers"])]
    if case["kind"] == "stack":
        return dict(kind="stack", stack=MoEStack(layers, routers, case["top_k"], eps=_EPS), h=_rows(case, seed))
    return dict(kind="block", block=MoEBlock(layers[0], case["top_k"]), h=_rows(case, seed), w=routers[0])


# ---- one pass ---------------------------------------------------------------------------------

def _product(s, p, x, y):
    m, (k, n) = x.shape[0], s["dims"][p]
    stream = torch.cuda.current_stream().cuda_stream
    if "scale" in s:
        capi.call("hm_matmul_w8a32", x.data_ptr(), s["w"][p].data_ptr(), s["scale"][p], 0, y.data_ptr(),
                  m, k, n, 0, s["scratch"].data_ptr(), s["scratch"].numel() * 4, stream)
    else:
        capi.call("hm_matmul_f32", x.data_ptr(), s["w"][p].data_ptr(), y.data_ptr(), m, k, n, stream)


def run(s):
    if s["kind"] == "stack":
        return s["stack"].launch(s["h"])
    if s["kind"] == "block":
        b = s["block"].launch(s["h"], s["w"])
        return {k: b[k] for k in _BLOCK_OUT}
    stream = torch.cuda.current_stream().cuda_stream
    _product(s, 0, s["x"], s["gate"])
    _product(s, 1, s["x"], s["up"])
    n = s["gate"].numel()
    capi.call("hm_silu", s["gate"].data_ptr(), s["act"].data_ptr(), n, stream)
    capi.call("hm_mul", s["act"].data_ptr(), s["up"].data_ptr(), s["z"].data_ptr(), n, stream)
    _product(s, 2, s["z"], s["y"])
    return {"gate": s["gate"], "up": s["up"], "z": s["z"], "y": s["y"]}


# ---- what a pass cannot do without ------------------------------------------------------------

def work(case):
    t, h, i, e, k = (case[n] for n in ("tokens", "hidden", "inter", "experts", "top_k"))
    size = 1 if case["dtype"] == "int8" else 4
    if case["kind"] == "ops":
        # three products, and two elementwise operations that each read and write whole rows
        return {"bytes": 3 * h * i * size + 4 * t * (3 * h + i * (2 + 2 + 3 + 1)), "flops": 6 * t * h * i}
    used = e * (1.0 - (1.0 - k / e) ** t)  # experts that at least one token picks
    pairs = t * k
    per_layer = used * 3 * h * i * size + 4 * h * e + 2 * 4 * t * h
    if case["kind"] == "block":
        per_layer += 4 * pairs * h + 4 * (4 * pairs + 2 * e)  # the expert rows and the routing results
    n = case["layers"]
    return {"bytes": n * per_layer, "flops": n * (6 * pairs * h * i + 2 * t * h * e)}


def tolerance(case):
    if case["kind"] == "ops":
        return {"rel": 1e-5}
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    # INT8 experts of more than 64 (token, expert) pairs read the activations as fixed-point digits
    # (two for the rows, three for the products): 5e-5 from the 64-bit result, a tenth of that once
    # the stack has added its residual; fewer pairs run in FP32 (4e-7 to 1.3e-6)
    if case["tokens"] * case["top_k"] > 64 or case["tokens"] > 16:
        return {"rel": 2e-5 if case["kind"] == "stack" else 2e-4}
    return {"rel": 1e-5}


# ---- the same in 64 bits ----------------------------------------------------------------------

def _exact_experts(x, ids, payload, scale, case):
    """[T, k, H]: every chosen expert's output for its token."""
    h, i = case["hidden"], case["inter"]
    y = torch.empty((x.shape[0], ids.shape[1], h), dtype=torch.float64, device="cuda")
    for e in range(case["experts"]):
        t, r = torch.nonzero(ids == e, as_tuple=True)
        if not len(t):
            continue
        w = payload[e].double()
        if scale is not None:
            w = w * scale[e].double()[:, None]
        g = x[t] @ w[0].view(h, i)
        u = x[t] @ w[1].view(h, i)
        y[t, r] = (g * torch.sigmoid(g) * u) @ w[2].view(i, h)
    return y


def _exact_block(x, case, seed, layer):
    payload, scale = _weights(case, seed, layer)
    logits = x @ _router(case, seed, layer).double()
    # ranked as the router ranks them: by the float32 logit, then by the lower expert
    ids = torch.sort(logits.float(), dim=1, descending=True, stable=True).indices[:, :case["top_k"]]
    scores = torch.softmax(logits, dim=1).gather(1, ids)
    scores = scores / scores.sum(dim=1, keepdim=True)
    y = _exact_experts(x, ids, payload, scale, case)
    return (scores[:, :, None] * y).sum(dim=1), ids, scores, y


def exact(case, seed):
    x = _rows(case, seed).double()
    if case["kind"] == "ops":
        q, scale = _weights(case, seed, 0)
        w = q[0].double() if scale is None else q[0].double() * scale[0].double()[:, None]
        h, i = case["hidden"], case["inter"]
        gate, up = x @ w[0].view(h, i), x @ w[1].view(h, i)
        z = gate * torch.sigmoid(gate) * up
        return {"gate": gate, "up": up, "z": z, "y": z @ w[2].view(i, h)}
    if case["kind"] == "stack":
        for n in range(case["layers"]):
            norm = x / torch.sqrt(x.square().mean(dim=1, keepdim=True) + float(np.float32(_EPS)))
            x = x + _exact_block(norm, case, seed, n)[0]
        return x
    out, ids, scores, y = _exact_block(x, case, seed, 0)
    order = torch.sort(ids.reshape(-1), stable=True).indices  # groups by expert, tokens ascending
    return {"out": out, "ids": None, "scores": scores, "counts": None, "offsets": None,
            "perm_tokens": None, "perm_weights": scores.reshape(-1)[order],
            "expert_out": y.reshape(-1, case["hidden"])[order]}
