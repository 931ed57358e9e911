"""Performance cases of the quantized-inference path, through its public entry points.

The work is what a program that serves or converts a quantized model calls:
quantized Linear layers in each of their five modes at decode, batched-decode
and prefill token counts, the INT4 FFN block, the multi-head attention layer
and the weight quantizers a conversion runs.  `listed()` holds the named cases,
`draw()` more of the same kinds over the ranges stated below.

Case fields by "kind":
  linear    mode (w4, w8, w8a8, fp8, fp8_weight), m tokens, n outputs, k inputs, bias
  mlp       m tokens, model width d, hidden width f (multiples of the INT4 group, 128)
  mha       mode (w4, w8), batch b, sequence s, h heads of width dh, causal mask or none
  quantize  op (i4, i8, fp8: a weight's codes and scales; i8_roundtrip: codes, scales and
            the dequantized copy; i4_dequant: codes back to f32; per_tensor: the
            asymmetric whole-tensor form of activation calibration), rows, k
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "neo-theano_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import theano_quantize as tq  # noqa: E402

# ranges of the drawn cases (the listed ones lie inside them)
M_RANGE = (1, 2048)        # tokens of a Linear or an FFN call
WIDTH_RANGE = (64, 16384)  # inputs and outputs of a layer
SEQ_RANGE = (1, 2048)
MAX_FLOPS = 3.4e11         # about the listed attention layer's
MAX_ELEMENTS = 14336 * 16384  # weight elements: about the largest listed projections


def listed():
    return [
        # one token through the widest INT4 projection of a 4096-wide model: single-stream decode
        {"name": "w4_decode", "kind": "linear", "mode": "w4", "m": 1, "n": 14336, "k": 4096, "bias": False},
        # the same for the default (INT8 weight-only) configuration's square projection: the smallest call
        {"name": "w8_decode", "kind": "linear", "mode": "w8", "m": 1, "n": 4096, "k": 4096, "bias": True},
        # a small decode batch through the FFN's down projection in the default configuration
        {"name": "w8_decode_down", "kind": "linear", "mode": "w8", "m": 4, "n": 4096, "k": 14336, "bias": False},
        # a prompt through the default configuration
        {"name": "w8_prefill", "kind": "linear", "mode": "w8", "m": 512, "n": 4096, "k": 4096, "bias": True},
        # a long prompt (or several) through INT8 weights and activations
        {"name": "w8a8_prefill", "kind": "linear", "mode": "w8a8", "m": 2048, "n": 4096, "k": 4096, "bias": False},
        # a decode batch of 64 streams on FP8, down projection
        {"name": "fp8_batch", "kind": "linear", "mode": "fp8", "m": 64, "n": 4096, "k": 14336, "bias": False},
        # a classifier head with a vocabulary and width that are no multiple of any tile
        {"name": "w8a8_ragged", "kind": "linear", "mode": "w8a8", "m": 77, "n": 1003, "k": 1000, "bias": True},
        # the FFN block of a 4096-wide model: decode batch and prompt
        {"name": "mlp_decode", "kind": "mlp", "m": 8, "d": 4096, "f": 14336},
        {"name": "mlp_prefill", "kind": "mlp", "m": 512, "d": 4096, "f": 14336},
        # the attention layer of the same model over a prompt of 2048 tokens
        {"name": "mha_prefill", "kind": "mha", "mode": "w4", "b": 1, "s": 2048, "h": 32, "dh": 128, "causal": False},
        # a small encoder/decoder layer on short, odd sequences, default configuration
        {"name": "mha_short", "kind": "mha", "mode": "w8", "b": 2, "s": 129, "h": 8, "dh": 64, "causal": True},
        # converting a checkpoint: the INT4 codes of one FFN weight
        {"name": "quantize_i4", "kind": "quantize", "op": "i4", "rows": 14336, "k": 4096},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, multiple):
    """A layer width: a multiple of 128 (as model widths are) half of the time, any otherwise."""
    w = _log(rng, *WIDTH_RANGE)
    step = max(multiple, 128 if rng.random() < 0.5 else 1)
    return min(WIDTH_RANGE[1], max(step, (w + step // 2) // step * step))


def draw(rng):
    kind = rng.choices(["linear", "mlp", "mha", "quantize"], [55, 15, 15, 15])[0]
    if kind == "linear":
        mode = rng.choice(["w4", "w8", "w8a8", "fp8", "fp8_weight"])
        n, k = _width(rng, 1), _width(rng, 128 if mode == "w4" else 1)
        while n * k > MAX_ELEMENTS:
            n = (n + 1) // 2
        m = min(_log(rng, *M_RANGE), max(1, int(MAX_FLOPS / (2 * n * k))))
        return {"kind": kind, "mode": mode, "m": m, "n": n, "k": k, "bias": rng.random() < 0.5}
    if kind == "mlp":
        d, f = 128 * _log(rng, 1, 64), 128 * _log(rng, 1, 128)
        m = min(_log(rng, *M_RANGE), max(1, int(MAX_FLOPS / (6 * d * f))))
        return {"kind": kind, "m": m, "d": d, "f": f}
    if kind == "mha":
        dh = rng.choice([32, 64, 64, 80, 96, 128, 128])
        h = 8 * rng.randint(1, 4)
        b, s = rng.randint(1, 4), _log(rng, *SEQ_RANGE)
        while b * s * (8 * (h * dh) ** 2 + 4 * s * h * dh) > MAX_FLOPS:
            s = (s + 1) // 2
        return {"kind": kind, "mode": rng.choice(["w4", "w8"]), "b": b, "s": s, "h": h, "dh": dh,
                "causal": rng.random() < 0.5}
    op = rng.choice(["i4", "i8", "fp8", "i8_roundtrip", "i4_dequant", "per_tensor"])
    rows, k = _log(rng, 1, 14336), _width(rng, 128 if op in ("i4", "i4_dequant") else 1)
    return {"kind": kind, "op": op, "rows": min(rows, max(1, 14336 * 4096 // k)), "k": k}


# ------------------------------------------------------------------ inputs
# Weights N(0, 0.02) and activations N(0, 1), as the repository's own measurements and tests take them.


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * int(seed) + 17)
    return g


def _normal(g, shape, std=1.0, dtype=torch.float32):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(std).to(dtype)


def _inputs(case, seed):
    """The raw tensors of a case: what the call takes, and the f32 weights behind its modules."""
    g, kind = _gen(seed), case["kind"]
    if kind == "linear":
        n, k = case["n"], case["k"]
        return {"w": _normal(g, (n, k), 0.02), "b": _normal(g, (n,), 0.1) if case["bias"] else None,
                "x": _normal(g, (case["m"], k), 1.0, torch.bfloat16 if case["mode"] == "w4" else torch.float32)}
    if kind == "mlp":
        d, f = case["d"], case["f"]
        return {"gate": _normal(g, (f, d), 0.02), "up": _normal(g, (f, d), 0.02), "down": _normal(g, (d, f), 0.02),
                "x": _normal(g, (case["m"], d), 1.0, torch.bfloat16)}
    if kind == "mha":
        e, s = case["h"] * case["dh"], case["s"]
        mask = None
        if case["causal"]:
            mask = torch.triu(torch.full((1, s, s), float("-inf"), device="cuda"), diagonal=1)
        return {"w": [_normal(g, (e, e), 0.02) for _ in range(4)], "b": [_normal(g, (e,), 0.1) for _ in range(4)],
                "x": _normal(g, (case["b"], s, e)), "mask": mask}
    return {"w": _normal(g, (case["rows"], case["k"]), 0.02)}


_CONFIGS = {
    "w4": tq.QConfig.default_int4,
    "w8": tq.QConfig.default_int8,
    "w8a8": lambda: tq.QConfig(tq.QuantDType.Int8, tq.QuantDType.Int8, True, True),
    "fp8": lambda: tq.QConfig(tq.QuantDType.FP8, tq.QuantDType.FP8, True, True),
    "fp8_weight": lambda: tq.QConfig(tq.QuantDType.FP8, tq.QuantDType.UInt8, True, True),
}

_QUANTIZERS = {
    "i4": tq.quantize_i4_g128,
    "i8": tq.quantize_per_channel_i8,
    "fp8": tq.quantize_per_channel_fp8,
    "i8_roundtrip": tq.fake_quantize_per_channel_i8,
    "per_tensor": lambda w: tq.quantize_per_tensor(w, tq.QuantDType.Int8),
}


def prepare(case, seed):
    r, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        return {"call": tq.QuantizedLinear.from_tensors(r["w"], r["b"], _CONFIGS[case["mode"]]()), "args": (r["x"],)}
    if kind == "mlp":
        return {"call": tq.QuantizedMLP.from_tensors(r["gate"], r["up"], r["down"]), "args": (r["x"],)}
    if kind == "mha":
        layer = tq.QuantizedMultiheadAttention.from_tensors(case["h"], *r["w"], *r["b"],
                                                            qconfig=_CONFIGS[case["mode"]]())
        return {"call": layer.forward_with_mask, "args": (r["x"], r["x"], r["x"], r["mask"])}
    if case["op"] == "i4_dequant":
        return {"call": tq.dequantize_i4_g128, "args": tuple(tq.quantize_i4_g128(r["w"]))}
    return {"call": _QUANTIZERS[case["op"]], "args": (r["w"],)}


def run(state):
    return state["call"](*state["args"])


# ------------------------------------------------------------------ the work
_ACT_BYTES = {"w4": 2}


def _weight_bytes(mode, n, k):
    return n * k // 2 + 2 * n * (k // 128) if mode == "w4" else n * k + 4 * n


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _weight_bytes(case["mode"], n, k) + m * k * _ACT_BYTES.get(case["mode"], 4) + 4 * m * n
                + (4 * n if case["bias"] else 0), "flops": 2 * m * n * k}
    if kind == "mlp":
        m, d, f = case["m"], case["d"], case["f"]
        return {"bytes": 3 * _weight_bytes("w4", d, f) + 6 * m * d, "flops": 6 * m * d * f}
    if kind == "mha":
        t, s, e = case["b"] * case["s"], case["s"], case["h"] * case["dh"]
        return {"bytes": 4 * _weight_bytes(case["mode"], e, e) + 16 * e + 8 * t * e + (4 * s * s if case["causal"] else 0),
                "flops": 8 * t * e * e + 4 * t * s * e}
    n, op = case["rows"] * case["k"], case["op"]
    if op in ("i4", "i4_dequant"):
        return {"bytes": 4 * n + n // 2 + 2 * (n // 128), "flops": 0}
    if op == "per_tensor":
        return {"bytes": 8 * n, "flops": 0}
    return {"bytes": (9 if op == "i8_roundtrip" else 5) * n + 4 * case["rows"], "flops": 0}


def tolerance(case):
    kind = case["kind"]
    # about four times what the path is off from 64 bits
    if kind == "linear":
        # w8a8 sums exactly and rounds in its epilogue only; the weight-only 8-bit modes sum in f32;
        # w4 sums each 128-long group in f32 with its scale applied afterwards; the FP8 matrix
        # instructions round inside their sums (1.5e-5 at K = 14336)
        return {"rel": {"w8a8": 3e-7, "w8": 2e-6, "fp8_weight": 2e-6, "w4": 2e-5, "fp8": 6e-5}[case["mode"]]}
    if kind == "mlp":
        return {"rel": 2e-5}  # the hidden activations are handed over as bf16 hi + lo, 2^-17 of each
    if kind == "mha":
        # w4 rounds the attention's output to bf16 before the last projection: a change of f32
        # rounding in the attention moves some of those values by one bf16 step
        return {"rel": 1e-3, "max": 2e-2} if case["mode"] == "w4" else {"rel": 1e-5}
    return "exact"


# ------------------------------------------------------------------ 64 bits
def _rhaz(v):
    return torch.sign(v) * torch.floor(v.abs() + 0.5)


def _row_scale(w, qmax):
    return (w.abs().amax(1, keepdim=True).double() / qmax).clamp_min(1e-10).float()


def _i8(w):
    s = _row_scale(w, 127.0)
    return _rhaz(w.double() / s.double()).clamp(-128, 127), s


def _fp8(w):
    s = _row_scale(w, 448.0)
    return (w.double() / s.double()).float().clamp(-448, 448).to(torch.float8_e4m3fn).double(), s


def _i4(w):
    n, k = w.shape
    g = w.view(n, k // 128, 128)
    s = (g.abs().amax(2, keepdim=True).double() / 7.0).float().half()
    s = torch.where(s == 0, torch.full_like(s, 2.0 ** -24), s)
    return _rhaz(g.double() / s.double()).clamp(-8, 7), s


def _dequantized(w, mode):
    q, s = {"w4": _i4, "w8": _i8, "w8a8": _i8, "fp8": _fp8, "fp8_weight": _fp8}[mode](w)
    return (q * s.double()).view(w.shape)


def _linear(x, w, b, mode):
    """x in f64 (already rounded to what the mode takes)."""
    if mode in ("w8a8", "fp8"):
        q, s = (_i8 if mode == "w8a8" else _fp8)(x.float())
        x = q * s.double()
    y = x @ _dequantized(w, mode).t().contiguous()
    return y if b is None else y + b.double()


def _attention(qkv, b, s, h, dh, mask):
    q, k, v = (t.reshape(b, s, h, dh).transpose(1, 2).contiguous() for t in qkv.split(h * dh, 1))
    out = torch.empty((b, s, h * dh), dtype=torch.float64, device=qkv.device)
    for i in range(b):
        for j in range(h):
            p = (q[i, j] @ k[i, j].t().contiguous()) / math.sqrt(dh)
            if mask is not None:
                p = p + mask[0].double()
            out[i, :, j * dh:(j + 1) * dh] = torch.softmax(p, -1) @ v[i, j]
    return out.view(b * s, h * dh)


def exact(case, seed):
    r, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        return _linear(r["x"].double(), r["w"], r["b"], case["mode"])
    if kind == "mlp":
        x = r["x"].double()
        g, u = (x @ _dequantized(r[n], "w4").t().contiguous() for n in ("gate", "up"))
        return (g / (1.0 + torch.exp(-g)) * u) @ _dequantized(r["down"], "w4").t().contiguous()
    if kind == "mha":
        mode, e = case["mode"], case["h"] * case["dh"]
        rounded = (lambda t: t.to(torch.bfloat16).double()) if mode == "w4" else (lambda t: t)
        x = rounded(r["x"].reshape(-1, e).double())
        qkv = torch.cat([_linear(x, r["w"][i], r["b"][i], mode) for i in range(3)], 1)
        o = rounded(_attention(qkv, case["b"], case["s"], case["h"], case["dh"], r["mask"]))
        return _linear(o, r["w"][3], r["b"][3], mode).view(case["b"], case["s"], e)
    w, op = r["w"], case["op"]
    if op == "i4_dequant":
        return _dequantized(w, "w4")
    if op == "per_tensor":
        lo, hi = w.min().double(), w.max().double()
        s = ((hi - lo) / 255.0).clamp_min(1e-10)
        z = _rhaz(-128.0 - lo / s).clamp(-128, 127)
        return _rhaz(w.double() / s + z).clamp(-128, 127), s, z
    if op == "i4":
        return None, _i4(w)[1].double().view(w.shape[0], -1)
    q, s = _fp8(w) if op == "fp8" else _i8(w)
    return (None, s.double().view(-1), q * s.double()) if op == "i8_roundtrip" else (None, s.double().view(-1))
