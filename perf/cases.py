"""The work that a user of this package has it do, as cases that can be timed.

Every case goes through the package's public entry points (esm_gfx950.Device
and esm_gfx950.Model, one call of the C ABI each):

  forward     a packed forward from host token ids: Model.forward_packed, or
              Model.forward_hidden_states where the hidden states are wanted
  attention   Device.attention_varlen: packed varlen attention, fp32 in and out
  linear_i8   Device.linear_i8: fp32 activations quantised, INT8 GEMM, bias
  ffn_up      Device.linear_i8_gelu_quant_r24: the W8A8 FFN's up-projection,
              GELU and the quantisation of the down-projection's input
  linear_f32  Device.linear_f32: the fp32 linear of the lm head and the 8M model

Models are the repository's ESM-2 shapes with its synthetic weights
(esm_gfx950.synthetic): the 8M model whole, the 650M and 3B ones with a few
of their 33 and 36 identical layers. Batches take the lengths of its
benchmark workloads: 16 sequences of 22-202 tokens, 8 of 256, 256 of 60-250
around 120, 64 spread evenly in the logarithm over 50-1024; and one sequence
alone. Models and weights are made once and kept, as a program keeps them;
token ids and activations come from the seed.
"""
from __future__ import annotations

import ctypes
import functools
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "esm-cpp_amd"))
import esm_gfx950 as eg  # noqa: E402
from esm_gfx950 import synthetic as syn  # noqa: E402

MODELS = {"8m": syn.ESM2_8M, "650m": syn.ESM2_650M, "3b": syn.ESM2_3B}
WEIGHT_SEED = 20261201
PRECISIONS = {"fp32": eg.ATTN_FP32, "bf16": eg.ATTN_BF16_MFMA, "f16x3": eg.ATTN_F16X3_MFMA}
MODES = {"token": eg.ACT_PER_TOKEN, "tensor": eg.ACT_PER_TENSOR}


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # One short protein through the whole 8M fp32 model, logits to the
        # host: the smallest call anyone makes, all launches and latency.
        {"name": "8m one sequence", "kind": "forward", "model": "8m", "layers": 6, "quant": "fp32", "out": "host",
         "dist": "uniform", "seqs": 1, "lo": 66, "hi": 66, "shape_seed": 1},
        # The 8M fp32 model on 16 sequences of 20-200 residues, logits kept on
        # the device.
        {"name": "8m batch", "kind": "forward", "model": "8m", "layers": 6, "quant": "fp32", "out": "device",
         "dist": "uniform", "seqs": 16, "lo": 22, "hi": 202, "shape_seed": 2},
        # Embeddings: every hidden state of the same kind of batch on the host.
        {"name": "8m hidden states", "kind": "forward", "model": "8m", "layers": 6, "quant": "fp32", "out": "hidden",
         "dist": "uniform", "seqs": 16, "lo": 22, "hi": 202, "shape_seed": 3},
        # One protein of ordinary length through 650M W8A8 layers: what an
        # interactive caller waits for.
        {"name": "650m one sequence", "kind": "forward", "model": "650m", "layers": 4, "quant": "token",
         "out": "device", "dist": "uniform", "seqs": 1, "lo": 301, "hi": 301, "shape_seed": 4},
        # The uniform 8 x 256 batch.
        {"name": "650m uniform batch", "kind": "forward", "model": "650m", "layers": 4, "quant": "token",
         "out": "device", "dist": "uniform", "seqs": 8, "lo": 256, "hi": 256, "shape_seed": 5},
        # The headline batch: 256 sequences of 60-250 tokens, about 31,000 in all.
        {"name": "650m varlen batch", "kind": "forward", "model": "650m", "layers": 4, "quant": "token",
         "out": "device", "dist": "normal", "seqs": 256, "lo": 60, "hi": 250, "shape_seed": 20261205},
        # The 3B shape on lengths spread over 50-1024 tokens.
        {"name": "3b long batch", "kind": "forward", "model": "3b", "layers": 2, "quant": "token", "out": "device",
         "dist": "log", "seqs": 64, "lo": 50, "hi": 1024, "shape_seed": 20261206},
        # The numerics that equal the x86 CPU path bit for bit (per-tensor
        # activation scales), as a check run of part of the headline batch.
        {"name": "650m x86-exact batch", "kind": "forward", "model": "650m", "layers": 2, "quant": "x86",
         "out": "device", "dist": "normal", "seqs": 64, "lo": 60, "hi": 250, "shape_seed": 8},
        # The facade's attention arm at the default numerics, ragged lengths.
        {"name": "attention f16x3", "kind": "attention", "precision": "f16x3", "heads": 20, "dist": "normal",
         "seqs": 64, "lo": 60, "hi": 250, "shape_seed": 9},
        # The facade's INT8 linear as its C++ host calls it: per-tensor
        # scales, the FFN up-projection's shape, an odd number of rows.
        {"name": "linear int8", "kind": "linear_i8", "mode": "tensor", "rows": 4099, "n": 5120, "k": 1280},
        # The default FFN up path of one large layer.
        {"name": "ffn up int8", "kind": "ffn_up", "rows": 15553, "n": 5120, "k": 1280},
        # The fp32 linear at the lm head's shape, an odd number of rows.
        {"name": "linear fp32", "kind": "linear_f32", "rows": 7777, "n": 1280, "k": 1280},
    ]


def draw(rng):
    """One more case of the listed ones' ranges."""
    def log(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(["8m", "8m", "650m", "650m", "650m", "3b", "x86", "attention", "linear_i8", "ffn_up",
                       "linear_f32"])
    shape_seed = rng.randrange(1 << 30)
    if kind in ("8m", "650m", "3b", "x86"):
        lo = log(22, 160)
        hi = min(1024, int(lo * math.exp(rng.uniform(0.0, 1.8))))
        tokens = log(lo, {"8m": 12000, "650m": 31000, "3b": 20000, "x86": 7500}[kind])
        if kind == "x86":
            hi = min(hi, 250)
            lo = min(lo, hi)
        seqs = max(1, min(256, int(tokens / math.sqrt(lo * hi))))
        return {"kind": "forward", "model": "650m" if kind == "x86" else kind,
                "layers": {"8m": 6, "650m": 4, "3b": 2, "x86": 2}[kind],
                "quant": {"8m": "fp32", "x86": "x86"}.get(kind) or rng.choice(["token", "token", "tensor"]),
                "out": rng.choice(["host", "device", "hidden"] if kind == "8m" else ["device", "device", "host"]),
                "dist": "log", "seqs": seqs, "lo": lo, "hi": hi, "shape_seed": shape_seed}
    if kind == "attention":
        precision = rng.choice(["f16x3", "f16x3", "bf16", "fp32"])
        lo = log(17, 160)
        hi = min(1024, int(lo * math.exp(rng.uniform(0.0, 1.8))))
        seqs = max(1, min(256, int(log(lo, 4000 if precision == "fp32" else 16000) / math.sqrt(lo * hi))))
        return {"kind": "attention", "precision": precision, "heads": rng.choice([20, 40]), "dist": "log",
                "seqs": seqs, "lo": lo, "hi": hi, "shape_seed": shape_seed}
    n, k = rng.choice([(1280, 1280), (3840, 1280), (5120, 1280), (1280, 5120), (2560, 2560)])
    if kind == "linear_i8":
        return {"kind": kind, "mode": rng.choice(["token", "tensor"]), "rows": log(30, 16000), "n": n, "k": k}
    if kind == "ffn_up":
        n, k = rng.choice([(5120, 1280), (5120, 1280), (10240, 2560)])
        return {"kind": kind, "rows": log(30, 31000 if k == 1280 else 15000), "n": n, "k": k}
    n, k = rng.choice([(320, 320), (960, 320), (1280, 320), (320, 1280), (1280, 1280), (1280, 1280), (2560, 2560)])
    return {"kind": "linear_f32", "rows": log(20, 16000), "n": n, "k": k}


def _lengths(case):
    """Token lengths of the case's sequences (the case's own, not the seed's)."""
    n, lo, hi = case["seqs"], case["lo"], case["hi"]
    if case["dist"] == "normal":
        return syn.varlen_lengths(n, case["shape_seed"], lo=lo, hi=hi)
    if case["dist"] == "log":
        return syn.loguniform_lengths(n, case["shape_seed"], lo=lo, hi=hi)
    return np.random.default_rng(case["shape_seed"]).integers(lo, hi + 1, size=n).astype(np.int32)


def _cu(lengths):
    cu = np.zeros(len(lengths) + 1, np.int32)
    cu[1:] = np.cumsum(lengths)
    return cu


# -------------------------------------------------- what a program keeps
@functools.lru_cache(None)
def _device():
    return eg.Device(0)


@functools.lru_cache(None)
def _weights(name, layers, int8):
    return syn.make_weights(MODELS[name].with_layers(layers), WEIGHT_SEED, int8=int8)


@functools.lru_cache(None)
def _model(name, layers, quant):
    int8 = quant != "fp32"
    m = eg.Model(_device(), _weights(name, layers, int8), int8=int8,
                 act_mode=eg.ACT_PER_TOKEN if quant == "token" else eg.ACT_PER_TENSOR,
                 attention_mode=eg.ATTN_MODE_F16X3)
    if quant == "x86":
        m.set_numerics(eg.NUMERICS_X86_AVX512)
    return m


@functools.lru_cache(None)
def _linear_weights(n, k):
    """(int8 codes, scales, bias) of an [n, k] linear, as numpy arrays."""
    rng = np.random.default_rng([WEIGHT_SEED, n, k])
    q, s = syn.quantize_weight(rng.standard_normal((n, k), dtype=np.float32) * np.float32(0.02))
    return q, s, rng.standard_normal(n, dtype=np.float32) * np.float32(0.02)


@functools.lru_cache(None)
def _weight_i8(n, k):
    return _device().weight_i8(*_linear_weights(n, k)[:2])


class _Dev:
    """A torch tensor as the entry points take it: a device pointer."""

    def __init__(self, t):
        self.t, self.ptr = t, ctypes.c_void_p(t.data_ptr())


def _empty(shape, dtype=torch.float32):
    return _Dev(torch.empty(shape, dtype=dtype, device="cuda"))


def _normal(seed, what, shape):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 16 + what)
    return torch.randn(shape, generator=g, device="cuda")


def _ids(case, seed):
    """cls, residues uniform over the 20 standard ones, eos, per sequence."""
    lengths = _lengths(case)
    cu = _cu(lengths)
    ids = np.random.default_rng([seed, 11]).integers(syn.RESIDUE_LO, syn.RESIDUE_HI + 1, size=int(cu[-1]),
                                                     dtype=np.int32)
    ids[cu[:-1]] = syn.CLS
    ids[cu[1:] - 1] = syn.EOS
    return ids, cu


def _activations(case, seed):
    """Rows as a LayerNorm leaves them: normal, each channel with a gain of
    its own, a few channels ten times the rest."""
    rows, k = case["rows"], case["k"]
    gain = torch.exp(0.3 * _normal(seed, 1, (k,)))
    gain[::97] *= 10.0
    return _normal(seed, 2, (rows, k)) * gain


def _quantize(x, per_row):
    """The activation rule, in fp32 as it is stated: scale = max|x| / 127 (1
    when all zero), code = clamp(rint(x * (1 / scale)))."""
    x = x.float()
    amax = x.abs().amax(dim=1, keepdim=True) if per_row else x.abs().max().reshape(1, 1)
    scale = torch.where(amax > 0, amax / 127.0, torch.ones_like(amax))
    return torch.clamp(torch.round(x * (1.0 / scale)), -127, 127), scale


# ------------------------------------------------------------ prepare and run
def prepare(case, seed):
    dev = _device()
    kind = case["kind"]
    s = {"dev": dev, "kind": kind}
    if kind == "forward":
        s["model"] = _model(case["model"], case["layers"], case["quant"])
        s["ids"], s["cu"] = _ids(case, seed)
        s["out"] = case["out"]
        if case["out"] == "device":
            s["logits"] = _empty((int(s["cu"][-1]), 33))
    elif kind == "attention":
        cu = _cu(_lengths(case))
        shape = (int(cu[-1]), case["heads"], 64)
        s.update(cu=cu, heads=case["heads"], precision=PRECISIONS[case["precision"]],
                 q=_Dev(_normal(seed, 1, shape) * 0.125), k=_Dev(_normal(seed, 2, shape)),
                 v=_Dev(_normal(seed, 3, shape)), y=_empty((shape[0], case["heads"] * 64)))
    elif kind == "linear_i8":
        m, n, k = case["rows"], case["n"], case["k"]
        s.update(m=m, n=n, k=k, mode=MODES[case["mode"]], x=_Dev(_activations(case, seed)), w=_weight_i8(n, k),
                 b=_Dev(torch.from_numpy(_linear_weights(n, k)[2]).cuda()), y=_empty((m, n)))
    elif kind == "ffn_up":
        m, n, k = case["rows"], case["n"], case["k"]
        codes, scale = _quantize(_activations(case, seed), True)
        s.update(m=m, n=n, k=k, x=_Dev(codes.to(torch.int8)), xs=_Dev(scale.reshape(m).contiguous()),
                 w=_weight_i8(n, k), b=_Dev(torch.from_numpy(_linear_weights(n, k)[2]).cuda()),
                 hi=_empty((m, n), torch.int16), lo=_empty((m + m % 2, n), torch.uint8),
                 y=_empty((m, n), torch.int8), ys=_empty((m,)))
    else:
        m, n, k = case["rows"], case["n"], case["k"]
        s.update(m=m, n=n, k=k, x=_Dev(_normal(seed, 1, (m, k))), w=_Dev(_normal(seed, 2, (n, k)) * 0.02),
                 b=_Dev(_normal(seed, 3, (n,)) * 0.02), y=_empty((m, n)))
    return s


def run(s):
    dev, kind = s["dev"], s["kind"]
    if kind == "forward":
        if s["out"] == "hidden":
            return list(s["model"].forward_hidden_states(s["ids"], s["cu"]))
        if s["out"] == "host":
            return s["model"].forward_packed(s["ids"], s["cu"])
        s["model"].forward_packed(s["ids"], s["cu"], s["logits"])
        return s["logits"].t
    if kind == "attention":
        dev.attention_varlen(s["q"], s["k"], s["v"], s["cu"], s["heads"], 64, s["y"], s["precision"])
        return s["y"].t
    if kind == "linear_i8":
        dev.linear_i8(s["x"], s["w"], s["b"], s["y"], s["m"], s["n"], s["k"], s["mode"])
        return s["y"].t
    if kind == "ffn_up":
        dev.linear_i8_gelu_quant_r24(s["x"], s["k"], s["xs"], s["w"], s["b"], s["m"], s["hi"], s["lo"], s["y"],
                                     s["n"], s["ys"])
        return [s["y"].t, s["ys"].t]
    dev.linear_f32(s["x"], s["w"], s["b"], s["y"], s["m"], s["n"], s["k"])
    return s["y"].t


# ------------------------------------------------------------ work and tolerance
def work(case):
    kind = case["kind"]
    if kind in ("forward", "attention"):
        lengths = _lengths(case).astype(np.float64)
        t, sq = float(lengths.sum()), float((lengths * lengths).sum())
    if kind == "forward":
        c = MODELS[case["model"]]
        d, f, layers = c.hidden_size, c.intermediate_size, case["layers"]
        per_layer, head = 4 * d * d + 2 * d * f, d * d + 33 * d
        size = 4 if case["quant"] == "fp32" else 1
        read = layers * per_layer * size + head * 4 + t * 4
        wrote = t * 33 * 4 + (t * d * 4 * (layers + 1) if case["out"] == "hidden" else 0)
        return {"bytes": read + wrote, "flops": 2 * t * (layers * per_layer + head) + 4 * sq * d * layers}
    if kind == "attention":
        return {"bytes": 4 * t * case["heads"] * 64 * 4, "flops": 4 * sq * case["heads"] * 64}
    m, n, k = case["rows"], case["n"], case["k"]
    flops = 2.0 * m * n * k
    if kind == "linear_i8":
        return {"bytes": 4 * m * k + n * k + 8 * n + 4 * m * n, "flops": flops}
    if kind == "ffn_up":
        return {"bytes": m * k + 4 * m + n * k + 8 * n + m * n + 4 * m, "flops": flops}
    return {"bytes": 4 * (m * k + n * k + n + m * n), "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind == "forward":
        if case["quant"] == "x86":
            return "exact"  # equal to the x86 CPU path bit for bit
        if case["quant"] == "fp32":
            return {"rel": 5e-6, "max": 3e-5}  # kernels in another order of sums: 1.4e-6, largest 6e-6
        # W8A8: every linear quantises its input again, so the last bit of a
        # sum in another order moves some int8 codes by one (scalar fp32
        # attention against split-fp16: 0.012-0.021, largest 0.065-0.113).
        return {"rel": 0.03, "max": 0.4}
    if kind == "attention":
        if case["precision"] == "bf16":
            return {"rel": 2e-3, "max": 2e-2}  # probabilities rounded to fp16
        return {"rel": 2e-6, "max": 4e-5}
    if kind == "linear_i8":
        return {"rel": 1e-6, "max": 1e-5}  # exact int32 sums, one fused step each
    if kind == "ffn_up":
        return {"rel": 1e-6, "max": 1e-5, "differ": 1e-4}  # codes next to a rounding tie
    return {"rel": 2e-6, "max": 4e-5}


# ------------------------------------------------------------------ 64 bits
def _f64(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda().double()


def _gelu64(x):
    return 0.5 * x * (1.0 + torch.erf(x / math.sqrt(2.0)))


def _round24(x):
    """The top 24 bits of the fp32 value (nearest, ties away from zero)."""
    return ((x.float().view(torch.int32) + 0x80) & -256).view(torch.float32).double()


def _layer_norm64(x, w, b, eps):
    x = x - x.mean(dim=1, keepdim=True)
    return x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + eps) * w + b


def _attention64(q, k, v, cu):
    """q, k, v [T, H, dh] float64 -> [T, H dh]."""
    out = torch.empty_like(q)
    for a, b in zip(cu[:-1].tolist(), cu[1:].tolist()):
        qs, ks, vs = (x[a:b].transpose(0, 1).contiguous() for x in (q, k, v))
        p = torch.softmax(torch.matmul(qs, ks.transpose(1, 2).contiguous()), dim=2)
        out[a:b] = torch.matmul(p, vs).transpose(0, 1)
    return out.reshape(q.shape[0], -1)


def _forward64(case, seed):
    c = MODELS[case["model"]].with_layers(case["layers"])
    d, heads, dh = c.hidden_size, c.num_heads, c.head_dim
    quant = case["quant"]
    w = _weights(case["model"], case["layers"], quant != "fp32")
    ids, cu = _ids(case, seed)
    lengths = cu[1:] - cu[:-1]

    def f(name):
        return _f64(w.f32[name])

    def linear(x, name, quantised=True):
        bias = f(name + ".bias")
        if quant == "fp32" or not quantised:
            return x @ f(name + ".weight").t() + bias
        codes, scale = _quantize(x, quant == "token")
        wq, ws = w.i8[name]
        return (codes.double() @ _f64(wq).t()) * (scale.double() * _f64(ws)[None, :]) + bias

    # Rotary tables from the fp32 angles that the model is defined with.
    half = dh // 2
    inv = np.float32(10000.0) ** (-(2 * np.arange(half, dtype=np.float32) / np.float32(dh)))
    pos = np.concatenate([np.arange(n) for n in lengths]).astype(np.float32)
    angle = _f64(pos[:, None] * inv[None, :].astype(np.float32))
    cos, sin = torch.cos(angle)[:, None, :], torch.sin(angle)[:, None, :]

    def rope(x):
        a, b = x[..., :half], x[..., half:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)

    hidden = f("embed")[torch.from_numpy(ids).cuda().long()] * (1.0 - 0.15 * 0.8)
    states = [hidden]
    for i in range(c.num_layers):
        p = "layers.%d." % i
        x = _layer_norm64(hidden, f(p + "attn_ln.weight"), f(p + "attn_ln.bias"), c.layer_norm_eps)
        q, k, v = (linear(x, p + n).reshape(-1, heads, dh) for n in ("q", "k", "v"))
        y = _attention64(rope(q / math.sqrt(dh)), rope(k), v, cu)
        hidden = hidden + linear(y, p + "out")
        x = _layer_norm64(hidden, f(p + "ffn_ln.weight"), f(p + "ffn_ln.bias"), c.layer_norm_eps)
        y = linear(x, p + "fc1")
        hidden = hidden + linear(_gelu64(_round24(y) if quant == "token" else y), p + "fc2")
        states.append(hidden)
    x = _layer_norm64(hidden, f("final_ln.weight"), f("final_ln.bias"), c.layer_norm_eps)
    states[-1] = x
    x = _gelu64(linear(x, "lm_head.dense", False))
    x = _layer_norm64(x, f("lm_head.ln.weight"), f("lm_head.ln.bias"), c.layer_norm_eps)
    logits = x @ f("embed").t() + f("lm_head.decoder.bias")
    return [logits, torch.stack(states)] if case["out"] == "hidden" else logits


def exact(case, seed):
    kind = case["kind"]
    if kind == "forward":
        return _forward64(case, seed)
    s = prepare(case, seed)
    if kind == "attention":
        return _attention64(s["q"].t.double(), s["k"].t.double(), s["v"].t.double(), s["cu"])
    if kind == "linear_f32":
        return s["x"].t.double() @ s["w"].t.double().t() + s["b"].t.double()
    wq, ws, b = _linear_weights(s["n"], s["k"])
    if kind == "linear_i8":
        codes, scale = _quantize(s["x"].t, case["mode"] == "token")
    else:
        codes, scale = s["x"].t, s["xs"].t.reshape(-1, 1)
    y = (codes.double() @ _f64(wq).t()) * (scale.double() * _f64(ws)[None, :]) + _f64(b)
    if kind == "linear_i8":
        return y
    return [None, _quantize(_gelu64(_round24(y)), True)[1].reshape(-1).double()]
