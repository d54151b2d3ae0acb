"""The work this library is timed on: the calls an inference engine makes
through inferno_hip, over the sizes it makes them at.

A case's "kind" is one path:

  gemv      one quantized matrix times one activation vector (any format)
  layers    the quantized decode work of several decoder layers: input norm +
            grouped wq/wk/wv, wo + residual, the FFN block with norm and
            residual.  Several layers, because a decode step walks a model's
            layers and meets every weight in memory, not in a cache
  lm_head   final norm, vocabulary projection, greedy token
  prefill   a batch of T tokens through one Q4_K weight, or through several
            weights that share the tokens (one rounding of X)
  prefill32 the same product on fp32 operands (the accurate option)
  int8      GEMV in the reference C library's int8-activation numerics
  dequant   blocks to fp32
  host      the drop-in q4_k_gemv! on host arrays, synchronous

Weights are packed from values shaped as quantizers leave them: quants spread
about the middle of their range, scales and mins such that the weights centre
on zero with a standard deviation of about 0.02.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parents[1] / "inferno.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from inferno_hip import QuantizedKernels as QK  # noqa: E402
from inferno_hip import device as D  # noqa: E402

Q8_0, Q4_K, Q5_K, Q6_K, IQ4_NL = 8, 12, 13, 14, 20
BYTES = {Q8_0: 34, Q4_K: 144, Q5_K: 176, Q6_K: 210, IQ4_NL: 18}
ELEMS = {Q8_0: 32, Q4_K: 256, Q5_K: 256, Q6_K: 256, IQ4_NL: 32}
GRID = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)
EPS = 1e-6


def listed():
    return [
        # a key or value projection on its own: the smallest decode call
        {"name": "gemv q4_k 1024x4096", "kind": "gemv", "type": Q4_K, "outer": 1024, "inner": 4096},
        # rows of no round number of columns, an odd number of rows
        {"name": "gemv q8_0 5003x2720", "kind": "gemv", "type": Q8_0, "outer": 5003, "inner": 2720},
        # one token through four layers of the benchmark's decoder (Q4_K, Q6_K down)
        {"name": "decode 4 layers 4096", "kind": "layers", "layers": 4, "hidden": 4096, "inter": 12288,
         "kv": 1024, "type": Q4_K, "down": Q6_K},
        # a smaller decoder, Q5_K throughout
        {"name": "decode 4 layers 2560 q5_k", "kind": "layers", "layers": 4, "hidden": 2560, "inter": 9728,
         "kv": 512, "type": Q5_K, "down": Q5_K},
        # the end of a decode step
        {"name": "lm_head q6_k 151936x2048", "kind": "lm_head", "type": Q6_K, "vocab": 151936, "hidden": 2048},
        # the benchmark's prompt length through one square projection
        {"name": "prefill 512x4096x4096", "kind": "prefill", "tokens": 512, "inner": 4096, "outers": "4096"},
        # a short prompt through gate and up
        {"name": "prefill 77x2560 gate/up", "kind": "prefill", "tokens": 77, "inner": 2560,
         "outers": "9728,9728"},
        # a long prompt through gate and up: the largest call
        {"name": "prefill 2048x4096 gate/up", "kind": "prefill", "tokens": 2048, "inner": 4096,
         "outers": "12288,12288"},
        # the accurate option at an odd prompt length
        {"name": "prefill32 509x2048x2048", "kind": "prefill32", "tokens": 509, "inner": 2048, "outer": 2048},
        # the reference C numerics on the FFN down projection
        {"name": "int8 q6_k 4096x12288", "kind": "int8", "type": Q6_K, "outer": 4096, "inner": 12288},
        # a weight unpacked for a path that wants fp32
        {"name": "dequant q6_k 4096x4096", "kind": "dequant", "type": Q6_K, "outer": 4096, "inner": 4096},
        # what a caller of q4_k_gemv! sees: host arrays in and out
        {"name": "host q4_k 4096x4096", "kind": "host", "outer": 4096, "inner": 4096},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def columns(t, lo, hi):
        e = ELEMS[t]
        return e * max(1, log_int(lo, hi) // e)

    any_type = (Q4_K, Q5_K, Q6_K, Q8_0, IQ4_NL)
    kind = rng.choice(("gemv", "gemv", "layers", "lm_head", "prefill", "prefill", "prefill", "prefill32", "int8",
                       "dequant", "host"))
    if kind == "gemv":
        t = rng.choice(any_type)
        return {"kind": kind, "type": t, "outer": log_int(512, 32768), "inner": columns(t, 1024, 16384)}
    if kind == "layers":
        hidden = 256 * rng.randint(4, 20)
        inter = 256 * int(hidden * rng.uniform(2.5, 4.0) / 256)
        t = rng.choice((Q4_K, Q4_K, Q5_K))
        return {"kind": kind, "layers": rng.randint(2, 4), "hidden": hidden, "inter": inter,
                "kv": 128 * rng.randint(2, 8), "type": t, "down": rng.choice((t, Q6_K))}
    if kind == "lm_head":
        return {"kind": kind, "type": rng.choice((Q6_K, Q6_K, Q8_0)), "vocab": rng.randint(32000, 152064),
                "hidden": 256 * rng.randint(4, 16)}
    if kind == "prefill":
        inner = columns(Q4_K, 1024, 14336)
        n = rng.choice((1, 1, 2, 3))
        most = 2048 * 4096 * 24576
        tokens = log_int(2, 2048)
        outers = []
        for _ in range(n):
            o = log_int(512, 14336)
            if rng.random() < 0.7:
                o = 256 * max(1, o // 256)
            outers.append(min(o, max(256, most // (n * tokens * inner))))
        return {"kind": kind, "tokens": tokens, "inner": inner, "outers": ",".join(map(str, outers))}
    if kind == "prefill32":
        return {"kind": kind, "tokens": log_int(8, 700), "inner": columns(Q4_K, 256, 4096),
                "outer": log_int(256, 4096)}
    if kind == "int8":
        t = rng.choice((Q4_K, Q5_K, Q6_K))
        return {"kind": kind, "type": t, "outer": log_int(512, 14336), "inner": columns(t, 1024, 14336)}
    if kind == "dequant":
        t = rng.choice(any_type)
        return {"kind": kind, "type": t, "outer": log_int(512, 12288), "inner": columns(t, 1024, 8192)}
    return {"kind": kind, "outer": log_int(512, 14336), "inner": columns(Q4_K, 1024, 14336)}


# ---- packed weights --------------------------------------------------------
def _half_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(-1, 2)


def _spread(g, shape, mid, dev, lo, hi):
    v = torch.randn(shape, generator=g, device="cuda") * dev + mid
    return v.round_().clamp_(lo, hi).to(torch.uint8)


def _pack_scales(sc, m):
    s = torch.empty((sc.shape[0], 12), dtype=torch.uint8, device=sc.device)
    s[:, 0:4] = sc[:, 0:4] | ((sc[:, 4:8] >> 4) << 6)
    s[:, 4:8] = m[:, 0:4] | ((m[:, 4:8] >> 4) << 6)
    s[:, 8:12] = (sc[:, 4:8] & 15) | ((m[:, 4:8] & 15) << 4)
    return s


def _blocks(g, t, n):
    """n blocks of format t, as one uint8 tensor."""
    vary = torch.exp(0.3 * torch.randn(n, generator=g, device="cuda"))
    b = torch.empty((n, BYTES[t]), dtype=torch.uint8, device="cuda")
    if t in (Q4_K, Q5_K):
        mid, dev, top = (7.5, 3.4, 15) if t == Q4_K else (15.5, 6.8, 31)
        d = vary * (0.02 / (42 * dev))
        b[:, 0:2] = _half_bytes(d)
        b[:, 2:4] = _half_bytes(d * mid)
        sc = torch.randint(20, 64, (n, 8), generator=g, device="cuda")
        m = (sc + torch.randint(-4, 5, (n, 8), generator=g, device="cuda")).clamp_(0, 63)
        b[:, 4:16] = _pack_scales(sc.to(torch.uint8), m.to(torch.uint8))
        q = _spread(g, (n, 4, 2, 32), mid, dev, 0, top)
        low = q & 15
        b[:, -128:] = (low[:, :, 0] | (low[:, :, 1] << 4)).reshape(n, 128)
        if t == Q5_K:
            hb = (q >> 4).reshape(n, 8, 32)
            qh = torch.zeros((n, 32), dtype=torch.uint8, device="cuda")
            for s in range(8):
                qh |= hb[:, s] << s
            b[:, 16:48] = qh
    elif t == Q6_K:
        q = _spread(g, (n, 2, 4, 32), 32, 12, 0, 63)
        b[:, 0:128] = torch.stack(((q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4),
                                   (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)), 2).reshape(n, 128)
        h = q >> 4
        b[:, 128:192] = (h[:, :, 0] | (h[:, :, 1] << 2) | (h[:, :, 2] << 4) | (h[:, :, 3] << 6)).reshape(n, 64)
        sc = torch.randint(40, 128, (n, 16), generator=g, device="cuda")
        sc = torch.where(torch.rand((n, 16), generator=g, device="cuda") < 0.5, -sc, sc)
        b[:, 192:208] = sc.to(torch.int8).view(torch.uint8)
        b[:, 208:210] = _half_bytes(vary * (0.02 / (84 * 12)) * 4)
    elif t == Q8_0:
        b[:, 0:2] = _half_bytes(vary * (0.02 / 42))
        q = torch.randn((n, 32), generator=g, device="cuda").mul_(42).round_().clamp_(-127, 127)
        b[:, 2:34] = q.to(torch.int8).view(torch.uint8)
    else:
        b[:, 0:2] = _half_bytes(vary * (0.02 / 60))
        q = _spread(g, (n, 2, 16), 7.5, 3.4, 0, 15)
        b[:, 2:18] = q[:, 0] | (q[:, 1] << 4)
    return b.reshape(-1)


def _weight(g, t, outer, inner):
    return D.DeviceWeight(_blocks(g, t, outer * (inner // ELEMS[t])), t, inner, outer)


def _half64(b2):
    return b2.contiguous().view(torch.float16).to(torch.float64)


def _unpack(data, t, outer, inner):
    """The matrix in 64 bits."""
    b = data.reshape(-1, BYTES[t])
    n = b.shape[0]
    if t in (Q4_K, Q5_K):
        d, dmin = _half64(b[:, 0:2]), _half64(b[:, 2:4])
        s = b[:, 4:16]
        sc = torch.cat((s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)), 1).to(torch.float64)
        m = torch.cat((s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)), 1).to(torch.float64)
        qs = b[:, -128:].reshape(n, 4, 32)
        q = torch.stack((qs & 15, qs >> 4), 2).reshape(n, 8, 32)
        if t == Q5_K:
            q = q | torch.stack([((b[:, 16:48] >> k) & 1) << 4 for k in range(8)], 1)
        w = (d * sc)[:, :, None] * q.to(torch.float64) - (dmin * m)[:, :, None]
    elif t == Q6_K:
        ql, qh = b[:, 0:128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 32)
        low = torch.stack((ql[:, :, 0] & 15, ql[:, :, 1] & 15, ql[:, :, 0] >> 4, ql[:, :, 1] >> 4), 2)
        high = torch.stack([(qh >> (2 * k)) & 3 for k in range(4)], 2)
        q = (low | (high << 4)).to(torch.float64) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).to(torch.float64)
        w = (_half64(b[:, 208:210]) * sc)[:, :, None] * q.reshape(n, 16, 16)
    elif t == Q8_0:
        w = _half64(b[:, 0:2]) * b[:, 2:34].contiguous().view(torch.int8).to(torch.float64)
    else:
        grid = torch.tensor(GRID, dtype=torch.float64, device=b.device)
        q = torch.cat((b[:, 2:18] & 15, b[:, 2:18] >> 4), 1)
        w = _half64(b[:, 0:2]) * grid[q.long()]
    return w.reshape(outer, inner)


def _act(g, *shape):
    """Activations: normal, with channels of different strength."""
    chan = torch.exp(0.4 * torch.randn(shape[-1], generator=g, device="cuda"))
    return torch.randn(shape, generator=g, device="cuda") * chan


def _norm_w(g, n):
    return torch.rand(n, generator=g, device="cuda") + 0.5


def _f32(n):
    return torch.empty(n, dtype=torch.float32, device="cuda")


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _outers(case):
    return [int(v) for v in case["outers"].split(",")]


# ---- the state a program keeps, and one pass -------------------------------
def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    s = {"case": case}
    if kind == "layers":
        hid, inter, t = case["hidden"], case["inter"], case["type"]
        s["x0"] = _act(g, hid)
        s["h"] = _f32(inter + hid)
        s["xn"] = _f32(hid)
        s["layers"] = [{
            "qkv": _weight(g, t, hid + 2 * case["kv"], hid), "wo": _weight(g, t, hid, hid),
            "wg": _weight(g, t, inter, hid), "wu": _weight(g, t, inter, hid),
            "wd": _weight(g, case["down"], hid, inter),
            "attn_norm": _norm_w(g, hid), "ffn_norm": _norm_w(g, hid), "attn": _act(g, hid),
            "qkv_out": _f32(hid + 2 * case["kv"]), "x": _f32(hid),
        } for _ in range(case["layers"])]
    elif kind in ("prefill", "prefill32"):
        T, inner = case["tokens"], case["inner"]
        outers = _outers(case) if kind == "prefill" else [case["outer"]]
        s["X"] = _act(g, T, inner)
        s["w"] = [_weight(g, Q4_K, o, inner) for o in outers]
        s["y"] = [torch.empty((T, o), dtype=torch.float32, device="cuda") for o in outers]
        if kind == "prefill":
            s["xh"] = D.prefill_scratch(T, inner)
    elif kind == "lm_head":
        s["w"] = _weight(g, case["type"], case["vocab"], case["hidden"])
        s["x"], s["nw"] = _act(g, case["hidden"]), _norm_w(g, case["hidden"])
        s["xn"], s["logits"], s["ws"] = _f32(case["hidden"]), _f32(case["vocab"]), D.ArgmaxWorkspace()
    elif kind == "dequant":
        s["w"] = _weight(g, case["type"], case["outer"], case["inner"])
        s["y"] = _f32(case["outer"] * case["inner"])
    elif kind == "host":
        s["w"] = _blocks(g, Q4_K, case["outer"] * case["inner"] // 256).cpu().numpy()
        s["x"] = _act(g, case["inner"]).cpu().numpy()
        s["y"] = np.empty(case["outer"], np.float32)
        # the weight is loaded on the first call that names it, as at a model's start
        QK.q4_k_gemv_(s["y"], s["w"], s["x"], case["inner"], case["outer"])
    else:
        s["w"] = _weight(g, case["type"], case["outer"], case["inner"])
        s["x"], s["y"] = _act(g, case["inner"]), _f32(case["outer"])
        if kind == "int8":
            s["q8"] = torch.empty(case["inner"] // 256 * QK.Q8_K_BYTES, dtype=torch.uint8, device="cuda")
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "gemv":
        return D.gemv(s["w"], s["x"], s["y"])
    if kind == "layers":
        x, outs = s["x0"], []
        for l in s["layers"]:
            D.gemv_norm(l["qkv"], l["attn_norm"], EPS, x, l["qkv_out"], s["xn"])
            D.gemv_add(l["wo"], l["attn"], x, l["x"])
            x = D.ffn_block(l["wg"], l["wu"], l["wd"], l["ffn_norm"], EPS, l["x"], s["h"])
            outs += [l["qkv_out"], x]
        return outs
    if kind == "lm_head":
        D.lm_head_argmax_norm(s["w"], s["nw"], EPS, s["x"], s["ws"], s["xn"], s["logits"])
        return [s["logits"], s["ws"].token]
    if kind == "prefill":
        if len(s["w"]) == 1:
            return [D.prefill_q4_k(s["w"][0], s["X"], s["y"][0], s["xh"])]
        D.prefill_convert(s["X"], s["xh"])
        return [D.prefill_q4_k_xh(w, s["xh"], case["tokens"], y) for w, y in zip(s["w"], s["y"])]
    if kind == "prefill32":
        return D.prefill_q4_k_f32(s["w"][0], s["X"], s["y"][0])
    if kind == "int8":
        return D.gemv_q8k_x(s["w"], s["x"], s["y"], s["q8"])
    if kind == "dequant":
        return D.dequantize(s["w"], s["y"])
    return QK.q4_k_gemv_(s["y"], s["w"], s["x"], case["inner"], case["outer"])


# ---- what a pass needs, and how close two correct ones are -----------------
def _matrix_bytes(t, outer, inner):
    return outer * (inner // ELEMS[t]) * BYTES[t]


def work(case):
    kind = case["kind"]
    if kind == "layers":
        hid, inter, t = case["hidden"], case["inter"], case["type"]
        rows = 2 * hid + 2 * case["kv"] + 2 * inter
        per = _matrix_bytes(t, rows, hid) + _matrix_bytes(case["down"], hid, inter) + 4 * (5 * hid + 2 * case["kv"])
        return {"bytes": case["layers"] * per, "flops": case["layers"] * 2 * (rows * hid + hid * inter)}
    if kind in ("prefill", "prefill32"):
        T, inner = case["tokens"], case["inner"]
        rows = sum(_outers(case)) if kind == "prefill" else case["outer"]
        return {"bytes": 4 * T * (inner + rows) + _matrix_bytes(Q4_K, rows, inner), "flops": 2 * T * rows * inner}
    if kind == "lm_head":
        return {"bytes": _matrix_bytes(case["type"], case["vocab"], case["hidden"]) + 4 * (2 * case["hidden"] + case["vocab"]),
                "flops": 2 * case["vocab"] * case["hidden"]}
    outer, inner = case["outer"], case["inner"]
    t = Q4_K if kind == "host" else case["type"]
    if kind == "dequant":
        return {"bytes": _matrix_bytes(t, outer, inner) + 4 * outer * inner, "flops": 2 * outer * inner}
    return {"bytes": _matrix_bytes(t, outer, inner) + 4 * (inner + outer), "flops": 2 * outer * inner}


def tolerance(case):
    kind = case["kind"]
    if kind in ("dequant", "int8"):
        return "exact"  # both are defined bit for bit
    if kind == "prefill":
        # fp16 operands: 7.5e-4 from 64 bits as measured at 77 to 2048 tokens
        return {"rel": 3e-3, "max": 2e-2}
    if kind == "layers":
        # fp32 sums through four layers: 5.2e-6 as measured
        return {"rel": 2e-5, "max": 2e-4}
    # fp32 sums: 1.9e-6 at most as measured
    return {"rel": 8e-6, "max": 8e-5}


# ---- the same in 64 bits ---------------------------------------------------
def _rmsnorm64(x, w):
    return x / torch.sqrt(torch.mean(x * x) + EPS) * w.double()


def _q8k64(x):
    """x as the int8 path rounds it: 256-value blocks, d = amax / 127, half away from zero."""
    v = x.reshape(-1, 256)
    d = v.abs().amax(1, keepdim=True) / 127.0
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    p = (v * inv).double()
    return (torch.sign(p) * torch.floor(p.abs() + 0.5) * d.double()).reshape(-1)


def exact(case, seed):
    s, kind = prepare(case, seed), case["kind"]

    def mat(w):
        return _unpack(w.data, w.ggml_type, w.outer, w.inner)

    if kind == "gemv":
        return mat(s["w"]) @ s["x"].double()
    if kind == "layers":
        x, outs = s["x0"].double(), []
        for l in s["layers"]:
            outs.append(mat(l["qkv"]) @ _rmsnorm64(x, l["attn_norm"]))
            x = x + mat(l["wo"]) @ l["attn"].double()
            n = _rmsnorm64(x, l["ffn_norm"])
            gate, up = mat(l["wg"]) @ n, mat(l["wu"]) @ n
            x = x + mat(l["wd"]) @ (gate / (1 + torch.exp(-gate)) * up)
            outs.append(x)
        return outs
    if kind == "lm_head":
        logits = mat(s["w"]) @ _rmsnorm64(s["x"].double(), s["nw"])
        return [logits, torch.argmax(logits).to(torch.int32).reshape(1)]
    if kind == "prefill":
        return [s["X"].double() @ mat(w).t().contiguous() for w in s["w"]]
    if kind == "prefill32":
        return s["X"].double() @ mat(s["w"][0]).t().contiguous()
    if kind == "int8":
        return mat(s["w"]) @ _q8k64(s["x"])
    if kind == "dequant":
        return mat(s["w"]).reshape(-1)
    w = _unpack(torch.from_numpy(s["w"]).cuda(), Q4_K, case["outer"], case["inner"])
    return (w @ torch.from_numpy(s["x"]).cuda().double()).cpu().numpy()
