"""Performance cases of libmxfp4hip: the work its users have it do, through its
public entry points (the mxfp4hip binding of the C ABI), on one MI355X.

What the listed cases stand for:

  decode_1      one token through an expert-sized MLP: the latency of a decode step
  decode_8      eight sequences decoded together through a dense model's MLP
  batch_40      a continuous batch of decoding sequences, past the GEMV's 16 tokens
  chunk_512     a prefill chunk through the expert-sized MLP
  prefill_4096  a long prompt through the dense MLP
  ragged_257    an odd token count and sizes that are multiples of 32 only
  w4a4_4096     prefill with FP4 activations, the largest MLP in use
  fp8_128       FP8 weights, a batch of 128
  w8a8_1000     INT8 weights and activations, an odd prefill length
  moe_256       64 experts and unevenly routed decode tokens
  matmul_1024   one MXFP4 projection on its own, f32 out
  quantize      f32 weights to MXFP4 when a model is loaded

draw() spreads over the same kinds of call: every MLP variant, weight format,
token count from one to the listed largest, and sizes on and off the tile grid.

Data: x ~ N(0, 1) in f16, weights ~ N(0, 0.02), quantized here in plain torch.
"""
import math
import os
import random
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "mpp-4.1-fp4-fp8-block_amd"))

import mxfp4hip as M  # noqa: E402

VARIANTS = {"fused": M.MLP_FUSED, "dequant": M.MLP_DEQUANT, "w4a4": M.MLP_W4A4, "scaled": M.MLP_SCALED}
FORMATS = {"fp8_e4m3": M.WFMT_FP8_E4M3, "fp8_e5m2": M.WFMT_FP8_E5M2, "int8": M.WFMT_INT8, "int4": M.WFMT_INT4,
           "w8a8": M.WFMT_W8A8}
MXFP4_GRID = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]

_dev = None


def device():
    """The library context that a program keeps for its life."""
    global _dev
    if _dev is None:
        _dev = M.Device(0)
    return _dev


# ---- the cases -------------------------------------------------------------------
def listed():
    return [
        {"name": "decode_1", "kind": "mlp", "weights": "fused", "tokens": 1, "hidden": 7168, "inter": 2048},
        {"name": "decode_8", "kind": "mlp", "weights": "fused", "tokens": 8, "hidden": 4096, "inter": 14336},
        {"name": "batch_40", "kind": "mlp", "weights": "fused", "tokens": 40, "hidden": 7168, "inter": 2048},
        {"name": "chunk_512", "kind": "mlp", "weights": "fused", "tokens": 512, "hidden": 7168, "inter": 2048},
        {"name": "prefill_4096", "kind": "mlp", "weights": "fused", "tokens": 4096, "hidden": 4096, "inter": 14336},
        {"name": "ragged_257", "kind": "mlp", "weights": "fused", "tokens": 257, "hidden": 2080, "inter": 5536},
        {"name": "w4a4_4096", "kind": "mlp", "weights": "w4a4", "tokens": 4096, "hidden": 8192, "inter": 28672},
        {"name": "fp8_128", "kind": "mlp", "weights": "fp8_e4m3", "tokens": 128, "hidden": 4096, "inter": 14336},
        {"name": "w8a8_1000", "kind": "mlp", "weights": "w8a8", "tokens": 1000, "hidden": 4096, "inter": 14336},
        {"name": "moe_256", "kind": "moe", "experts": 64, "tokens": 256, "hidden": 7168, "inter": 2048},
        {"name": "matmul_1024", "kind": "matmul", "a": "f16", "c": "f32", "m": 1024, "n": 4096, "k": 4096},
        {"name": "quantize", "kind": "quantize", "src": "f32", "rows": 14336, "k": 4096},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, lo, hi, step):
    return max(step, int(_log(rng, lo, hi)) // step * step)


def draw(rng):
    kind = rng.choices(["mlp", "moe", "matmul", "quantize"], [8, 2, 2, 1])[0]
    if kind == "mlp":
        weights = rng.choice(["fused"] * 5 + ["dequant", "w4a4", "scaled"] + sorted(FORMATS))
        # the fused, dequant and weight-format rows take any multiple of 32
        step = {"w4a4": 256, "scaled": 128, "w8a8": 128}.get(weights) or rng.choice([32, 64, 128, 128, 256])
        tokens = max(1, int(_log(rng, 1, 4097)))
        hidden, inter = _size(rng, 1024, 8192, step), _size(rng, 2048, 16384, step)
        return {"kind": kind, "weights": weights, "tokens": tokens, "hidden": hidden, "inter": inter}
    if kind == "moe":
        experts = rng.choice([8, 16, 32, 64])
        return {"kind": kind, "experts": experts, "tokens": int(_log(rng, experts, 4096)),
                "hidden": _size(rng, 1024, 7168, 128), "inter": _size(rng, 1024, 2048, 128)}
    if kind == "matmul":
        n = _size(rng, 512, 16384, 64) if rng.random() < 0.7 else int(_log(rng, 512, 16384))
        return {"kind": kind, "a": rng.choice(["f16", "f16", "f32"]), "c": rng.choice(["f32", "f16"]),
                "m": max(1, int(_log(rng, 1, 4096))), "n": n, "k": _size(rng, 1024, 8192, rng.choice([32, 128]))}
    return {"kind": kind, "src": rng.choice(["f32", "f16"]), "rows": int(_log(rng, 16, 28672)),
            "k": _size(rng, 1024, 16384, 32)}


def counts_of(case):
    """Rows of each expert: a router's uneven load (some experts several times
    as popular as others), the same for every seed."""
    e, t = case["experts"], case["tokens"]
    rng = random.Random(e * 100003 + t)
    share = [math.exp(rng.gauss(0.0, 0.6)) for _ in range(e)]
    got = [0] * e
    for i in rng.choices(range(e), share, k=t):
        got[i] += 1
    return got


# ---- weights in plain torch ---------------------------------------------------------
def _codes_mxfp4(v):
    """f32 [..., 32 n] -> (codes uint8 [..., 32 n], E8M0 bytes [..., n]):
    scale 2^(floor(log2 amax) - 2), nearest E2M1 value, ties to even."""
    b = v.reshape(*v.shape[:-1], -1, 32)
    amax = b.abs().amax(-1)
    e = torch.where(amax > 0, torch.frexp(amax)[1] - 3, torch.zeros_like(amax, dtype=torch.int32)).clamp(-127, 127)
    m = torch.ldexp(b, -e.unsqueeze(-1)).abs()
    code = torch.zeros(m.shape, dtype=torch.uint8, device=v.device)
    for i, at in enumerate([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0]):
        code += (m > at) if i % 2 == 0 else (m >= at)
    code |= (b < 0).to(torch.uint8) << 3
    return code.reshape(v.shape), (e + 127).to(torch.uint8)


def _pack4(code):
    return code[..., 0::2] | code[..., 1::2] << 4


def _unpack4(packed):
    return torch.stack([packed & 15, packed >> 4], -1).reshape(*packed.shape[:-1], -1)


def _mxfp4_f64(code, e8):
    grid = torch.tensor(MXFP4_GRID + [-g for g in MXFP4_GRID], dtype=torch.float64, device=code.device)
    v = grid[code.int()].reshape(*e8.shape, 32)
    return torch.ldexp(v, (e8.int() - 127).unsqueeze(-1)).reshape(code.shape)


def _rows(n, k):
    """Row ranges of about 64 M values, so that temporaries stay small."""
    step = max(1, (64 << 20) // k)
    return [(r, min(n, r + step)) for r in range(0, n, step)]


def _weights(fmt, n, k, gen):
    """(data, scales) of one random matrix [n][k] in a weight format."""
    parts = []
    for lo, hi in _rows(n, k):
        w = torch.randn(hi - lo, k, device="cuda", generator=gen) * 0.02
        if fmt == "int4":
            b = w.reshape(hi - lo, k // 32, 32)
            s = (b.abs().amax(-1) / 7.0).half()
            code = (b / s.float().unsqueeze(-1)).round().clamp(-8, 7).to(torch.int8).view(torch.uint8) & 15
            parts.append((_pack4(code.reshape(hi - lo, k)), s))
        elif fmt in ("fp8_e4m3", "fp8_e5m2"):
            top, dt = (448.0, torch.float8_e4m3fn) if fmt == "fp8_e4m3" else (57344.0, torch.float8_e5m2)
            s = w.abs().amax(-1, keepdim=True) / top
            parts.append(((w / s).to(dt).view(torch.uint8), s.reshape(-1)))
        elif fmt in ("int8", "w8a8"):
            s = w.abs().amax(-1, keepdim=True) / 127.0
            parts.append(((w / s).round().clamp(-127, 127).to(torch.int8).view(torch.uint8), s.reshape(-1)))
        else:
            code, e8 = _codes_mxfp4(w)
            parts.append((_pack4(code), e8))
    if len(parts) == 1:
        return parts[0]
    return torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts])


def _weights_f64(fmt, data, scales):
    if fmt == "int4":
        v = _unpack4(data).to(torch.int8)
        v = ((v ^ 8) - 8).double().reshape(*scales.shape, 32) * scales.double().unsqueeze(-1)
        return v.reshape(data.shape[0], -1)
    if fmt in ("fp8_e4m3", "fp8_e5m2"):
        dt = torch.float8_e4m3fn if fmt == "fp8_e4m3" else torch.float8_e5m2
        return data.view(dt).double() * scales.double().unsqueeze(-1)
    if fmt in ("int8", "w8a8"):
        return data.view(torch.int8).double() * scales.double().unsqueeze(-1)
    return _mxfp4_f64(_unpack4(data), scales)


# ---- inputs ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _shapes(case):
    return ((case["inter"], case["hidden"]), (case["inter"], case["hidden"]), (case["hidden"], case["inter"]))


def _inputs(case, seed):
    """The tensors of one call, from the seed alone."""
    g = _gen(seed)
    kind = case["kind"]
    if kind in ("mlp", "moe"):
        e = case.get("experts", 1)
        fmt = case.get("weights", "fused")
        x = torch.randn(case["tokens"], case["hidden"], device="cuda", generator=g).half()
        return {"x": x, "w": [_weights(fmt, e * n, k, g) for n, k in _shapes(case)]}
    if kind == "matmul":
        a = torch.randn(case["m"], case["k"], device="cuda", generator=g)
        return {"a": a.half() if case["a"] == "f16" else a, "w": [_weights("fused", case["n"], case["k"], g)]}
    w = torch.randn(case["rows"], case["k"], device="cuda", generator=g) * 0.02
    return {"w": w.half() if case["src"] == "f16" else w}


def _buf(t):
    return M.DevBuf(device(), t.data_ptr(), t.numel() * t.element_size())


def prepare(case, seed):
    s = dict(_inputs(case, seed), case=case)
    kind = case["kind"]
    if kind in ("mlp", "moe"):
        s["out"] = torch.empty(case["tokens"], case["hidden"], dtype=torch.float16, device="cuda")
        s["args"] = (_buf(s["x"]), M.Device.weights(*[(_buf(d), _buf(e)) for d, e in s["w"]]), _buf(s["out"]))
        if kind == "moe":
            s["counts"] = counts_of(case)
    elif kind == "matmul":
        s["out"] = torch.empty(case["m"], case["n"], dtype=torch.float32 if case["c"] == "f32" else torch.float16,
                               device="cuda")
        s["args"] = (_buf(s["a"]), _buf(s["w"][0][0]), _buf(s["out"]), _buf(s["w"][0][1]))
    else:
        s["packed"] = torch.empty(case["rows"], case["k"] // 2, dtype=torch.uint8, device="cuda")
        s["scales"] = torch.empty(case["rows"], case["k"] // 32, dtype=torch.uint8, device="cuda")
        s["args"] = (_buf(s["w"]), _buf(s["packed"]), _buf(s["scales"]))
    torch.cuda.synchronize()  # the library works on a stream of its own
    return s


def run(s):
    case, dev, args = s["case"], device(), s["args"]
    kind = case["kind"]
    if kind == "mlp":
        x, w, out = args
        if case["weights"] in FORMATS:
            dev.fmt_mlp_forward(FORMATS[case["weights"]], case["tokens"], case["hidden"], case["inter"], x, w, out)
        else:
            dev.mlp_forward(VARIANTS[case["weights"]], case["tokens"], case["hidden"], case["inter"], x, w, out)
        return s["out"]
    if kind == "moe":
        x, w, out = args
        dev.moe_forward(case["hidden"], case["inter"], s["counts"], x, w, out)
        return s["out"]
    if kind == "matmul":
        a, b, c, e8 = args
        dev.mxfp4_matmul(a, M.DT_F16 if case["a"] == "f16" else M.DT_F32, b, c,
                         M.DT_F32 if case["c"] == "f32" else M.DT_F16, case["m"], case["n"], case["k"], e8)
        return s["out"]
    src, packed, scales = args
    dev.mxfp4_quantize(src, M.DT_F16 if case["src"] == "f16" else M.DT_F32, case["rows"], case["k"], packed, scales)
    return [s["packed"], s["scales"]]


# ---- what a pass cannot do without --------------------------------------------------------
def _matrix_bytes(fmt, n, k):
    if fmt == "int4":
        return n * k // 2 + n * (k // 32) * 2
    if fmt in FORMATS:
        return n * k + n * 4
    return n * k // 2 + n * k // 32


def work(case):
    kind = case["kind"]
    if kind in ("mlp", "moe"):
        t, h, i = case["tokens"], case["hidden"], case["inter"]
        used = sum(c > 0 for c in counts_of(case)) if kind == "moe" else 1
        w = used * sum(_matrix_bytes(case.get("weights", "fused"), n, k) for n, k in _shapes(case))
        return {"bytes": w + 2 * t * h * 2, "flops": 6 * t * h * i}
    if kind == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _matrix_bytes("fused", n, k) + m * k * (2 if case["a"] == "f16" else 4)
                + m * n * (4 if case["c"] == "f32" else 2), "flops": 2 * m * n * k}
    n, k = case["rows"], case["k"]
    return {"bytes": n * k * (2 if case["src"] == "f16" else 4) + _matrix_bytes("fused", n, k), "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    if kind == "matmul":
        return {"rel": 1e-5 if case["c"] == "f32" else 1e-3}
    fmt = case.get("weights", "fused")
    if fmt == "w4a4":
        return {"rel": 4e-3}
    if fmt == "w8a8":
        return {"rel": 2e-3}
    if fmt == "scaled":
        return {"rel": 4e-3}
    return {"rel": 1e-3}


# ---- 64 bits ----------------------------------------------------------------------------
def _int8_rows(v):
    # the format's scale is an f32, and f16 values meet its ties often: the
    # codes are those of f32 division, as the format says
    v = v.float()
    s = v.abs().amax(-1, keepdim=True) / 127.0
    s = torch.where(s > 0, s, torch.ones_like(s))
    return (v / s).round().clamp(-127, 127).double() * s.double()


def _mxfp4_rows(v):
    code, e8 = _codes_mxfp4(v)
    return _mxfp4_f64(code, e8)


def _mlp_f64(fmt, x, mats):
    # the formats' own activations: FP4 or INT8, for x and for the middle
    act = {"w4a4": _mxfp4_rows, "w8a8": _int8_rows}.get(fmt, lambda v: v)
    x = act(x.double())
    g = x @ _weights_f64(fmt, *mats[0]).T
    u = x @ _weights_f64(fmt, *mats[1]).T
    mid = act(g / (1.0 + torch.exp(-g)) * u)
    return mid @ _weights_f64(fmt, *mats[2]).T


def exact(case, seed):
    kind = case["kind"]
    if kind == "quantize":
        return None
    s = _inputs(case, seed)
    if kind == "matmul":
        return s["a"].double() @ _weights_f64("fused", *s["w"][0]).T
    if kind == "mlp":
        return _mlp_f64(case["weights"], s["x"], s["w"])
    out, at = [], 0
    for e, c in enumerate(counts_of(case)):
        mats = [(d[e * n:(e + 1) * n], q[e * n:(e + 1) * n]) for (d, q), (n, _) in zip(s["w"], _shapes(case))]
        if c:
            out.append(_mlp_f64("fused", s["x"][at:at + c], mats))
        at += c
    return torch.cat(out)
