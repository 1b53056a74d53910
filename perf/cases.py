"""Performance cases of the integer Mamba inference path on one GPU.

Each case is one call (or one short run of calls) that a program using this
framework makes through its public entry points: the drop-in modules
(``MambaIntegerModel``, ``MambaIntegerBlock``, ``MambaIntegerBlockV2``,
``BitLinear``, ``DyadicScanFunction``, ``ssd_chunked_scan_forward``), the scan
ops of ``mamba_int.ops`` and the runner's prefill and greedy decode.  The sizes
are those of ``bench.py`` and the tests (d768 x 24, d2048 x 48, the multi-head
SSD block of the shipped config, the single-layer scan and BitLinear shapes)
and odd ones between them.

The whole path is integer arithmetic with frozen rounding rules, so every
output, the float ones included (an int32 times one float32 scale), is the same
bits on every correct implementation: every tolerance is "exact".
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mamba-integer_amd"))

from mamba_int import ModelDims, init_random_params, ops  # noqa: E402
from mamba_int.model import DecodeState, random_device_params  # noqa: E402
from mamba_integer_model import (DyadicScanFunction, MambaIntegerBlock, MambaIntegerBlockV2,  # noqa: E402
                                 MambaIntegerModel)
from rational_bitnet import BitLinear  # noqa: E402
from ssd_chunked_scan import ssd_chunked_scan_forward  # noqa: E402

DEV = "cuda:0"
SHIFT = 15


def listed():
    return [
        # one selective-scan layer of a short prompt: the smallest scan call
        {"name": "scan_layer", "kind": "scan", "batch": 1, "len": 256, "d": 512, "n": 16},
        # the long-context multi-head scan (24 heads of 64, 128 states, 8192 steps)
        {"name": "ssd_scan_long", "kind": "ssd_scan", "batch": 4, "len": 8192, "heads": 24, "head_dim": 64, "n": 128,
         "chunk": 256},
        # DyadicScanFunction over the materialized [B, L, d_inner * d_state] input of a d768 block
        {"name": "elementwise_scan", "kind": "elementwise", "batch": 1, "len": 2048, "channels": 24576},
        # the chunked scan's drop-in over d_inner channels, a length that no chunk divides
        {"name": "chunked_scan", "kind": "chunked", "batch": 4, "len": 1000, "channels": 1536, "chunk": 64},
        # a BitLinear projection of a prefill (float in, float out)
        {"name": "bitlinear_prefill", "kind": "bitlinear", "rows": 4096, "k": 768, "n": 3072, "bias": False},
        # a BitLinear with ragged sizes and a bias over a few tokens: the smallest layer call
        {"name": "bitlinear_ragged", "kind": "bitlinear", "rows": 37, "k": 1000, "n": 1108, "bias": True},
        # one dyadic block over a ragged batch of prompts, float hidden states in and out
        {"name": "block_ragged", "kind": "block", "block": "dyadic", "batch": 3, "len": 701, "d": 1024},
        # one multi-head SSD block of the shipped config
        {"name": "ssd_block", "kind": "block", "block": "ssd", "batch": 2, "len": 1023, "d": 768},
        # scoring: float logits of every position
        {"name": "model_forward", "kind": "forward", "batch": 2, "len": 1000, "d": 768, "layers": 24},
        # the prompt half of a generation: last-position logits and the recurrent state
        {"name": "model_prefill", "kind": "prefill", "batch": 8, "len": 2048, "d": 768, "layers": 24},
        # greedy decode of a small batch (chained step graphs), then the logits that follow
        {"name": "decode_b8", "kind": "decode", "block": "dyadic", "batch": 8, "steps": 64, "d": 768, "layers": 24},
        # greedy decode of the wide model at a serving batch
        {"name": "decode_wide_b64", "kind": "decode", "block": "dyadic", "batch": 64, "steps": 16, "d": 2048,
         "layers": 48},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["scan", "ssd_scan", "elementwise", "chunked", "bitlinear", "bitlinear", "block", "block",
                       "forward", "prefill", "decode", "decode"])
    if kind == "scan":
        return {"kind": kind, "batch": _log(rng, 1, 16), "len": _log(rng, 16, 2048), "d": 16 * _log(rng, 4, 128),
                "n": rng.choice([16, 32, 64])}
    if kind == "ssd_scan":
        return {"kind": kind, "batch": rng.randint(1, 4), "len": _log(rng, 64, 8192), "heads": _log(rng, 2, 24),
                "head_dim": rng.choice([32, 48, 64]), "n": rng.choice([16, 32, 64, 128]),
                "chunk": rng.choice([64, 128, 256])}
    if kind == "elementwise":
        c = _log(rng, 512, 24576)
        return {"kind": kind, "batch": rng.randint(1, max(1, min(8, 24576 // c))), "len": _log(rng, 32, 2048),
                "channels": c}
    if kind == "chunked":
        return {"kind": kind, "batch": _log(rng, 1, 8), "len": _log(rng, 32, 2048), "channels": _log(rng, 512, 2048),
                "chunk": rng.choice([16, 64, 100, 256])}
    if kind == "bitlinear":
        return {"kind": kind, "rows": _log(rng, 1, 4096), "k": _log(rng, 256, 2048), "n": 4 * _log(rng, 64, 768),
                "bias": rng.random() < 0.5}
    if kind == "block":
        if rng.random() < 0.4:
            return {"kind": kind, "block": "ssd", "batch": _log(rng, 1, 8), "len": _log(rng, 16, 2048), "d": 768}
        return {"kind": kind, "block": "dyadic", "batch": _log(rng, 1, 8), "len": _log(rng, 16, 2048),
                "d": 64 * _log(rng, 4, 16)}
    if kind == "forward":
        return {"kind": kind, "batch": _log(rng, 1, 4), "len": _log(rng, 16, 1000), "d": 64 * rng.randint(6, 12),
                "layers": rng.randint(4, 24)}
    if kind == "prefill":
        return {"kind": kind, "batch": _log(rng, 1, 8), "len": _log(rng, 32, 2048), "d": 64 * rng.randint(6, 12),
                "layers": rng.randint(4, 24)}
    if rng.random() < 0.3:
        return {"kind": kind, "block": "ssd", "batch": _log(rng, 1, 16), "steps": rng.randint(2, 32), "d": 768,
                "layers": rng.randint(2, 6)}
    return {"kind": kind, "block": "dyadic", "batch": _log(rng, 1, 64), "steps": rng.randint(2, 32),
            "d": rng.choice([384, 512, 768, 1024, 1536, 2048]), "layers": rng.randint(4, 24)}


# ------------------------------------------------------------------ programs
def _dims(c):
    if c.get("block") == "ssd":
        # the shipped config: 24 heads of 64 channels, 64 states, vocab 4096
        return ModelDims(d_model=c["d"], n_layer=c["layers"], vocab_size=4096, d_state=64, dt_rank=0, block="ssd",
                         n_heads=24, d_head=64)
    return ModelDims(d_model=c["d"], n_layer=c["layers"], vocab_size=32000, d_state=16, dt_rank=_dt_rank(c["d"]))


def _dt_rank(d):
    return -(-d // 256) * 16     # d_model / 16 rounded up to the packing unit


@functools.lru_cache(maxsize=2)
def _model(d, layers, block):
    """The model a serving program keeps: random weights, one for all prompts."""
    dims = _dims({"d": d, "layers": layers, "block": block})
    params = init_random_params(dims, 3) if dims.ssd else random_device_params(dims, 3, DEV)
    ssm = {"d_state": dims.d_state, "dt_rank": dims.dt_rank, "use_ssd": dims.ssd, "n_heads": 24, "d_head": 64}
    config = {"d_model": d, "n_layer": layers, "vocab_size": dims.vocab_size, "ssm_cfg": ssm}
    return MambaIntegerModel(config, params=params)


@functools.lru_cache(maxsize=2)
def _block(d, block):
    config = {"d_model": d, "n_layer": 24, "vocab_size": 32000,
              "ssm_cfg": {"d_state": 16, "dt_rank": _dt_rank(d)} if block == "dyadic"
              else {"d_state": 64, "n_heads": 24, "d_head": 64, "use_ssd": True}}
    return (MambaIntegerBlock if block == "dyadic" else MambaIntegerBlockV2)(config, 0, seed=3)


@functools.lru_cache(maxsize=2)
def _linear(k, n, bias):
    g = torch.Generator().manual_seed(3)
    layer = BitLinear(k, n, bias=bias)
    with torch.no_grad():
        layer.weight.copy_(torch.randn(n, k, generator=g) / math.sqrt(k))
        if bias:
            layer.bias.copy_(torch.randn(n, generator=g) * 0.1)
    layer = layer.to(DEV)
    layer(torch.zeros(1, k, device=DEV))     # the packed weights, laid out once
    return layer


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 7919 + 17)
    return g


def _ints(g, lo, hi, shape, dtype):
    return torch.randint(lo, hi + 1, shape, generator=g, device=DEV, dtype=torch.int32).to(dtype)


def prepare(case, seed):
    c, g, kind = case, _gen(seed), case["kind"]
    s = {"case": c}
    if kind == "scan":
        s["x"] = _ints(g, -127, 127, (c["batch"], c["len"], c["d"]), torch.int8)
        s["b"], s["c"] = (_ints(g, -127, 127, (c["batch"], c["len"], c["n"]), torch.int8) for _ in range(2))
        s["decay"] = _ints(g, 16384, 32767, (c["d"], c["n"]), torch.int32)
    elif kind == "ssd_scan":
        s["x"] = _ints(g, -127, 127, (c["batch"], c["len"], c["heads"], c["head_dim"]), torch.int8)
        s["b"], s["c"] = (_ints(g, -127, 127, (c["batch"], c["len"], c["heads"], c["n"]), torch.int8)
                          for _ in range(2))
        s["decay"] = _ints(g, 24576, 32767, (c["heads"],), torch.int32)
    elif kind in ("elementwise", "chunked"):
        shape = (c["batch"], c["len"], c["channels"])
        s["u"] = _ints(g, -100000, 100000, shape, torch.int32)
        s["nums"] = _ints(g, 16384, 32000, shape, torch.int32)
    elif kind == "bitlinear":
        s["layer"] = _linear(c["k"], c["n"], c["bias"])
        s["x"] = torch.randn(c["rows"], c["k"], generator=g, device=DEV)
    elif kind == "block":
        s["layer"] = _block(c["d"], c["block"])
        s["x"] = torch.randn(c["batch"], c["len"], c["d"], generator=g, device=DEV) * 4.0
    else:
        s["model"] = model = _model(c["d"], c["layers"], c.get("block", "dyadic"))
        run = model.runner(DEV)
        length = c.get("len", 16)
        s["ids"] = _ints(g, 0, run.dims.vocab_size - 1, (c["batch"], length), torch.int64)
        if kind == "decode":
            # a prompt has been read: its last logits and recurrent state (the
            # layers' states are rows of two tensors, which run() returns)
            D, N, n = run.dims.d_inner, run.dims.d_state, c["layers"]
            s["conv"] = torch.zeros((n, c["batch"], 3, D), dtype=torch.int8, device=DEV)
            s["h"] = torch.zeros((n, c["batch"], D, N), dtype=torch.int32, device=DEV)
            s["state"] = DecodeState(list(s["conv"].unbind(0)), list(s["h"].unbind(0)))
            s["logits"], _ = run.prefill(s["ids"], s["state"])
            # a server's warm-up: the step graphs of a batch are captured once
            warm = model.__dict__.setdefault("_warmed", set())
            if (c["batch"], c["steps"]) not in warm:
                run.decode_loop(s["logits"], s["state"].clone(), c["steps"])
                warm.add((c["batch"], c["steps"]))
    return s


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "scan":
        return ops.dyadic_scan(s["x"], s["b"], s["c"], s["decay"], SHIFT)
    if kind == "ssd_scan":
        return ops.ssd_chunked_scan(s["x"], s["b"], s["c"], s["decay"], SHIFT, c["chunk"])
    if kind == "elementwise":
        return DyadicScanFunction.apply(s["u"], s["nums"], SHIFT)
    if kind == "chunked":
        return ssd_chunked_scan_forward(s["u"], s["nums"], SHIFT, c["chunk"])
    if kind in ("bitlinear", "block"):
        return s["layer"](s["x"])
    if kind == "forward":
        return s["model"](s["ids"])
    runner = s["model"].runner(DEV)
    if kind == "prefill":
        logits, state = runner.prefill(s["ids"])
        return {"logits": logits, "state": state.h, "conv": state.conv}
    tokens = runner.decode_loop(s["logits"], s["state"], c["steps"])
    logits = runner.decode_step(tokens[:, -1].contiguous(), s["state"])
    return {"tokens": tokens, "logits": logits, "h": s["h"], "conv": s["conv"]}


# ---------------------------------------------------------------- accounting
def _layer_work(dims, rows, batch):
    """(weight and parameter bytes, state bytes written once, operations) of one
    layer over `rows` tokens of `batch` sequences."""
    d, D, N, X = dims.d_model, dims.d_inner, dims.d_state, dims.xp_width
    macs = 2 * D * d + X * D + d * D + (0 if dims.ssd else D * dims.dt_rank)
    params = macs // 4 + 8 * D + 2 * d + (dims.n_heads * 255 * 4 if dims.ssd else D * N * 4)
    state = batch * (D * N * 4 + 3 * D)
    return params, state, rows * (2 * macs + 4 * D * N)


def work(case):
    c, kind = case, case["kind"]
    if kind in ("scan", "ssd_scan"):
        h, p = (1, c["d"]) if kind == "scan" else (c["heads"], c["head_dim"])
        rows = c["batch"] * c["len"]
        return {"bytes": rows * h * (5 * p + 2 * c["n"]) + (p * c["n"] if kind == "scan" else h) * 4,
                "flops": 4 * rows * h * p * c["n"]}
    if kind == "elementwise":
        e = c["batch"] * c["len"] * c["channels"]
        return {"bytes": 12 * e, "flops": 2 * e}
    if kind == "chunked":
        e = c["batch"] * c["len"] * c["channels"]
        return {"bytes": 12 * e + 8 * c["batch"] * -(-c["len"] // c["chunk"]) * c["channels"], "flops": 3 * e}
    if kind == "bitlinear":
        m, k, n = c["rows"], c["k"], c["n"]
        return {"bytes": 4 * m * k + k * n // 4 + 4 * m * n, "flops": 2 * m * k * n}
    if kind == "block":
        dims = _dims(dict(c, layers=1))
        rows = c["batch"] * c["len"]
        params, _, flops = _layer_work(dims, rows, c["batch"])
        return {"bytes": params + 8 * rows * c["d"], "flops": flops}
    dims = _dims(c)
    head = dims.vocab_size * dims.d_model
    b = c["batch"]
    if kind == "decode":
        params, state, flops = _layer_work(dims, b, b)
        step = {"bytes": c["layers"] * (params + 2 * state) + head // 4 + b * dims.d_model,
                "flops": c["layers"] * flops + 2 * b * head}
        # the loop makes steps - 1 recurrent steps, and one more gives the logits
        return {"bytes": c["steps"] * step["bytes"] + 4 * b * dims.vocab_size, "flops": c["steps"] * step["flops"]}
    rows = b * c["len"]
    params, state, flops = _layer_work(dims, rows, b)
    out = rows if kind == "forward" else b
    return {"bytes": c["layers"] * (params + (state if kind == "prefill" else 0)) + head // 4 +
            rows * (8 + dims.d_model) + 4 * out * dims.vocab_size,
            "flops": c["layers"] * flops + 2 * out * head}


def tolerance(case):
    return "exact"


# ------------------------------------------------- the float outputs in 64 bits
def _rshr(v, s):
    return (v + (1 << (s - 1))) >> s if s > 0 else v


def _isqrt(v):
    r = torch.sqrt(v.double()).to(torch.int64)
    r = torch.where(r * r > v, r - 1, r)
    return torch.where((r + 1) * (r + 1) <= v, r + 1, r)


def _t64(a):
    return torch.as_tensor(np.asarray(a.cpu()) if isinstance(a, torch.Tensor) else np.asarray(a)).to(DEV).to(torch.int64)


def _matmul(a, packed):
    """Exact integer a @ W^T of a 2-bit packed ternary W (words of 16 weights,
    weight 4j + i at bits 8i + 2j)."""
    p = _t64(packed)
    q = torch.arange(16, device=DEV)
    byte = p.reshape(p.shape[0], -1, 4)[..., q & 3]
    code = (byte >> (2 * (q >> 2))) & 3
    w = torch.where(code >= 2, code - 4, code).reshape(p.shape[0], -1).double()
    return torch.round(a.double() @ w.t()).to(torch.int64)


def _norm64(r, gamma, v2):
    d = r.shape[-1]
    x = r - torch.div(r.sum(-1, keepdim=True), d, rounding_mode="floor")
    S = (x * x).sum(-1, keepdim=True)
    k = sum((S >= d * 4 ** (j + 8)).long() for j in range(1, 7 if v2 else 9)) - \
        sum((S < d * 4 ** (8 - j)).long() for j in range(1, 3 if v2 else 4))
    sh = 12 + k
    return ((x * _t64(gamma) + (torch.ones_like(sh) << (sh - 1))) >> sh).clamp(-127, 127)


def _block64(ly, dims, r):
    """One integer block over int64 residual rows r [B, L, d]."""
    B, L, d = r.shape
    D, N = dims.d_inner, dims.d_state
    xz = _rshr(_matmul(_norm64(r, ly.gamma, dims.ssd), ly.w_in), ly.s_in).clamp(-127, 127)
    x, z = xz[..., :D], xz[..., D:]
    xp = torch.cat([x.new_zeros(B, 3, D), x], 1)
    cw = _t64(ly.conv_w)
    v = (_t64(ly.conv_b) + sum(cw[:, j] * xp[:, j:j + L] for j in range(4))).clamp(-51200, 51200)
    xs = _rshr(v + _isqrt(v * v + (1 << 22)), 7).clamp(-127, 127)
    p = _rshr(_matmul(xs, ly.w_x), ly.s_x).clamp(-127, 127)
    y = torch.empty(B, L, D, dtype=torch.int64, device=DEV)
    if dims.ssd:
        H, P = dims.n_heads, dims.d_head
        bc = p[..., :2 * H * N].reshape(B, L, 2, H, N)
        S = (bc * bc).sum(-1, keepdim=True)
        inv = torch.where(S > 0, (1 << 30) // _isqrt(S << 16).clamp(min=1), 0)
        q = _rshr(bc * inv, 15).clamp(-127, 127)
        tab = _t64(ly.decay_tab)
        dec = tab[torch.arange(H, device=DEV), p[..., 2 * H * N:2 * H * N + H] + 127]
        h = torch.zeros(B, H, P, N, dtype=torch.int64, device=DEV)
        xh = xs.reshape(B, L, H, P)
        for t in range(L):
            h = (((h * dec[:, t, :, None, None]) >> 15) + q[:, t, 0, :, None, :] * xh[:, t, :, :, None]
                 ).clamp(-2**31, 2**31 - 1)
            y[:, t] = (h * q[:, t, 1, :, None, :]).sum(-1).reshape(B, D)
        y = y.clamp(-2**31, 2**31 - 1).clamp(-100 << 18, 100 << 18)
    else:
        R = dims.dt_rank
        dm = _rshr(_matmul(p[..., :R], ly.w_dt), ly.s_dt).clamp(-20, 20)
        sq = (dm * 65536 + _isqrt(dm * dm * (1 << 32) + (1 << 34))) >> 1
        xd = _rshr(xs * _rshr(655 * sq, 16).clamp(66, 6554), 10)
        Bm, Cm, base = p[..., R:R + N], p[..., R + N:R + 2 * N], _t64(ly.base)
        h = torch.zeros(B, D, N, dtype=torch.int64, device=DEV)
        for t in range(L):
            n = (base + dm[:, t, :, None]).clamp(0, 32000)
            h = (((h * n) >> 15) + Bm[:, t, None, :] * xd[:, t, :, None]).clamp(-2**31, 2**31 - 1)
            y[:, t] = (h * Cm[:, t, None, :]).sum(-1)
        y = y.clamp(-2**31, 2**31 - 1)
    gate = 16384 + torch.sign(z) * ((16384 * z.abs()) // (16 + z.abs()))
    yo = _rshr((y * gate) >> 15, ly.s_y).clamp(-127, 127)
    acc = _matmul(yo, ly.w_out)
    if ly.out_clamp > 0:
        acc = acc.clamp(-ly.out_clamp, ly.out_clamp)
    return (r + _rshr(acc * ly.res_mult, ly.res_shift)).clamp(-(2**23 - 1), 2**23 - 1)


def exact(case, seed):
    """The float outputs of run() in 64 bits; the others are whole numbers that
    are compared bit for bit."""
    kind = case["kind"]
    if kind not in ("chunked", "bitlinear", "block", "forward"):
        return None
    s = prepare(case, seed)
    if kind == "chunked":
        nums, cs = s["nums"].to(torch.int64), case["chunk"]
        ends, p = [], None
        for t in range(case["len"]):
            p = torch.full_like(nums[:, 0], 1 << 30) if t % cs == 0 else p
            p = (p * nums[:, t]) >> SHIFT
            if (t + 1) % cs == 0 or t + 1 == case["len"]:
                ends.append(p.double() / 2**30)
        return (None, None, torch.stack(ends, 1))
    if kind == "bitlinear":
        # the quantizer's IEEE float32 formula is the layer's definition; the
        # product and its scale are taken in 64 bits
        w, x = s["layer"].weight.detach().cpu(), s["x"].cpu()
        ws = torch.clamp(w.abs().mean(), min=1e-6)
        wq = torch.clamp(torch.round(w / ws), -1, 1).double()
        amax = torch.clamp(x.abs().amax(-1, keepdim=True), min=1e-8)
        xq = torch.clamp(torch.round(x * torch.div(torch.full_like(amax, 127.0), amax)), -127, 127).double()
        y = (xq.to(DEV) @ wq.to(DEV).t()) * (ws.double() * (amax.double() / 127.0)).to(DEV)
        return y + s["layer"].bias.detach().double() if case["bias"] else y
    if kind == "block":
        layer = s["layer"]
        r = torch.round(s["x"] * 256.0).clamp(-(2**23 - 1), 2**23 - 1).to(torch.int64)
        return _block64(layer.params, layer.dims, r).double() / 256.0
    model = s["model"]
    params = model.params
    r = _t64(params.emb)[s["ids"]] << 4
    for ly in params.layers:
        r = _block64(ly, model.dims, r)
    return _matmul(_norm64(r, params.gamma_f, False), params.w_head).double() * model.logit_scale
