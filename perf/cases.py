"""The calls this library is measured on: the quantised and bf16 linear layers
and the mixture-of-experts blocks of a transformer, each through the public
entry points, from one decode token to a long prefill.

``listed()`` holds the named calls, ``draw`` gives further calls of the same
kinds and ranges.  A kind is one way a program uses the library:

  mxfp4    dynamic MXFP4 quant of a bf16 activation, then ``gemm_a4w4``
  mxfp8    ``gemm_a8w4_mxfp8_dynamic`` (MXFP8 activation, MXFP4 weight)
  bf16     ``tgemm.mm`` (row-major or preshuffled weight, bf16 or f32 output)
  norm     residual add + RMSNorm + MXFP4 quant in one op, then ``gemm_a4w4``
  batched  ``batched_gemm_bf16_CK`` (one small weight per head)
  moe      ``fused_moe`` with MXFP4 weights

Weights are quantised and laid out once, in ``prepare``, as a program does at
load time; activations, routing and residuals come fresh with the state.
"""
from __future__ import annotations

import math

import torch

import aiter_amd

BF16_LIMIT = 4001 * 4096 * 14336       # M * N * K of the largest bf16 call
MXFP4_LIMIT = 8192 * 8192 * 8192
MXFP8_LIMIT = 2048 * 7168 * 16384
WEIGHT_LIMIT = 8192 * 28672            # N * K
MOE_PAIRS = 3000 * 9                   # tokens * topk
MOE_WEIGHT = 257 * 7168 * 256          # experts * model_dim * inter_dim

# (N, K) of the layers that bench.py sweeps and the tests run
LAYERS = [(7168, 2048), (4096, 4096), (14336, 4096), (4096, 14336), (7168, 16384), (28672, 8192), (8192, 28672)]
# (experts, topk, model_dim, inter_dim) of the MoE models in bench.py that fit the limits
MOE_SHAPES = [(257, 9, 7168, 256), (256, 8, 3072, 256), (512, 10, 4096, 256)]


def listed():
    return [
        # one decode token through an output projection: latency and launches
        {"name": "mxfp4_1_token", "kind": "mxfp4", "m": 1, "n": 7168, "k": 2048, "round": "even", "bias": False},
        # a ragged decode batch through a long-K down projection with a bias
        {"name": "mxfp4_67_tokens", "kind": "mxfp4", "m": 67, "n": 4096, "k": 14336, "round": "up", "bias": True},
        # a long prefill through a square layer, the largest MXFP4 product
        {"name": "mxfp4_8192_tokens", "kind": "mxfp4", "m": 8192, "n": 8192, "k": 8192, "round": "even",
         "bias": False},
        # a decode batch with MXFP8 activations, a ragged number of rows
        {"name": "mxfp8_300_tokens", "kind": "mxfp8", "m": 300, "n": 7168, "k": 16384},
        # expert scores of a decode batch: a thin bf16 product with f32 output
        {"name": "bf16_router_24_tokens", "kind": "bf16", "m": 24, "n": 256, "k": 7168, "out": "f32", "bias": False,
         "preshuffled": False},
        # a chunk of prefill mixed with decode through an up projection
        {"name": "bf16_150_tokens", "kind": "bf16", "m": 150, "n": 14336, "k": 4096, "out": "bf16", "bias": False,
         "preshuffled": False},
        # a ragged prefill through a down projection, the largest bf16 product
        {"name": "bf16_4001_tokens", "kind": "bf16", "m": 4001, "n": 4096, "k": 14336, "out": "bf16", "bias": False,
         "preshuffled": False},
        # the entry of a block in prefill: residual, norm, quant, projection
        {"name": "norm_1777_tokens", "kind": "norm", "m": 1777, "n": 6144, "k": 4096},
        # per-head projections of a decode batch
        {"name": "batched_16x100", "kind": "batched", "b": 16, "m": 100, "n": 1024, "k": 4096, "bias": False},
        # expert blocks: two decode tokens, a decode batch, a prefill
        {"name": "moe_2_tokens", "kind": "moe", "m": 2, "experts": 257, "topk": 9, "dim": 7168, "inter": 256,
         "act": "silu"},
        {"name": "moe_100_tokens", "kind": "moe", "m": 100, "experts": 257, "topk": 9, "dim": 7168, "inter": 256,
         "act": "silu"},
        {"name": "moe_3000_tokens", "kind": "moe", "m": 3000, "experts": 257, "topk": 9, "dim": 7168, "inter": 256,
         "act": "silu"},
    ]


def _log_int(rng, lo, hi, step=1):
    """A multiple of ``step`` in [lo, hi], evenly spread over the logarithm."""
    lo, hi = max(lo, step), max(hi, step)
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step)) // step * step


def _layer(rng, n_step, k_step, n_lo=512, n_hi=16384, k_lo=512, k_hi=28672):
    """(N, K): a layer of the sweep, or any other within the weight limit."""
    if rng.random() < 0.4:
        return rng.choice(LAYERS)
    n = _log_int(rng, n_lo, n_hi, n_step)
    return n, _log_int(rng, k_lo, min(k_hi, WEIGHT_LIMIT // n), k_step)


def draw(rng):
    kind = rng.choice(["mxfp4", "mxfp4", "mxfp8", "bf16", "bf16", "norm", "batched", "moe", "moe"])
    if kind == "mxfp4":
        n, k = _layer(rng, 16, 256)
        return {"kind": kind, "m": _log_int(rng, 1, min(8192, MXFP4_LIMIT // (n * k))), "n": n, "k": k,
                "round": rng.choice(["even", "up"]), "bias": rng.random() < 0.25}
    if kind == "mxfp8":
        n, k = _layer(rng, 16, 256)
        return {"kind": kind, "m": _log_int(rng, 1, min(4096, MXFP8_LIMIT // (n * k))), "n": n, "k": k}
    if kind == "bf16":
        if rng.random() < 0.2:
            return {"kind": kind, "m": _log_int(rng, 1, 4096), "n": _log_int(rng, 32, 512, 16),
                    "k": _log_int(rng, 1024, 8192, 64), "out": "f32", "bias": False, "preshuffled": False}
        n, k = _layer(rng, 16, 64)
        return {"kind": kind, "m": _log_int(rng, 1, min(4096, BF16_LIMIT // (n * k))), "n": n, "k": k,
                "out": "bf16", "bias": rng.random() < 0.25, "preshuffled": rng.random() < 0.3}
    if kind == "norm":
        n, k = _layer(rng, 16, 256, k_hi=8192)
        k = min(k, 8192)
        return {"kind": kind, "m": _log_int(rng, 1, min(8192, MXFP4_LIMIT // (n * k))), "n": n, "k": k}
    if kind == "batched":
        b, n = _log_int(rng, 4, 64), _log_int(rng, 128, 2048, 16)
        k = _log_int(rng, 128, 4096, 64)
        return {"kind": kind, "b": b, "m": _log_int(rng, 1, max(1, min(1024, BF16_LIMIT // (4 * b * n * k)))), "n": n,
                "k": k, "bias": rng.random() < 0.25}
    if rng.random() < 0.5:
        experts, topk, dim, inter = rng.choice(MOE_SHAPES)
    else:
        experts, topk = _log_int(rng, 8, 256), rng.randint(1, 8)
        dim = _log_int(rng, 1024, 7168, 256)
        inter = _log_int(rng, 256, min(2048, max(256, MOE_WEIGHT // (experts * dim))), 256)
    # pairs * inter_dim bounds the products, pairs the rows that are summed
    most = min(MOE_PAIRS, MOE_PAIRS * 256 * 7168 // (inter * dim)) // topk
    return {"kind": "moe", "m": _log_int(rng, 1, max(1, min(4096, most))), "experts": experts, "topk": topk,
            "dim": dim, "inter": inter, "act": rng.choice(["silu", "silu", "gelu"])}


# ------------------------------------------------------------------ inputs
def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 16 + salt)


def _activations(seed, shape, salt=0):
    """bf16 activations: normal, with the few strong channels that hidden
    states have (one in 128, 8 times the rest)."""
    g = _gen(seed, salt)
    x = torch.randn(shape, device="cuda", dtype=torch.bfloat16, generator=g)
    strong = torch.rand(shape[-1], device="cuda", generator=g) < 1 / 128
    return x * torch.where(strong, 8.0, 1.0).to(torch.bfloat16)


def _weights(seed, shape, salt=1):
    """bf16 weights, normal with a standard deviation of 2^-6."""
    return torch.randn(shape, device="cuda", dtype=torch.bfloat16, generator=_gen(seed, salt)).mul_(0.015625)


def _vector(seed, n, salt):
    return torch.randn(n, device="cuda", generator=_gen(seed, salt))


def _routing(case, seed):
    """Softmax top-k routing of random scores with uneven expert popularity."""
    g = _gen(seed, 3)
    e = case["experts"]
    scores = torch.randn(case["m"], e, device="cuda", generator=g) + 0.3 * torch.randn(e, device="cuda", generator=g)
    w, ids = torch.topk(torch.softmax(scores, -1), min(case["topk"], e), -1)
    return (w / w.sum(-1, keepdim=True)).contiguous(), ids.to(torch.int32).contiguous()


def _mxfp4_weight(w):
    """Packed, preshuffled MXFP4 rows and their shuffled scales."""
    q, s = aiter_amd.dynamic_mxfp4_quant(w, shuffle=True)
    return aiter_amd.shuffle_weight(q), s


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "moe":
        e, dim, inter = case["experts"], case["dim"], case["inter"]
        w1, st["w1_scale"] = _mxfp4_weight(_weights(seed, (e * 2 * inter, dim), 1))
        w2, st["w2_scale"] = _mxfp4_weight(_weights(seed, (e * dim, inter), 2))
        st["w1"], st["w2"] = w1.view(e, 2 * inter, dim // 2), w2.view(e, dim, inter // 2)
        st["topk_weight"], st["topk_ids"] = _routing(case, seed)
        st["x"] = _activations(seed, (case["m"], dim))
        return st
    if kind == "batched":
        st["x"] = _activations(seed, (case["b"], case["m"], case["k"]))
        st["w"] = _weights(seed, (case["b"], case["n"], case["k"]))
        st["bias"] = _vector(seed, case["n"], 2).expand(case["b"], -1).contiguous() if case["bias"] else None
        return st
    st["x"] = _activations(seed, (case["m"], case["k"]))
    w = _weights(seed, (case["n"], case["k"]))
    if kind == "bf16":
        st["w"] = aiter_amd.shuffle_weight(w) if case["preshuffled"] else w
    else:
        st["w"], st["w_scale"] = _mxfp4_weight(w)
    if kind == "norm":
        st["residual"] = _activations(seed, (case["m"], case["k"]), 4)
        st["gamma"] = (1 + 0.1 * _vector(seed, case["k"], 5)).to(torch.bfloat16)
    st["bias"] = _vector(seed, case["n"], 2) if case.get("bias") else None
    return st


EPS = 1e-6


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "mxfp4":
        quant = aiter_amd.get_hip_quant if case["round"] == "up" else aiter_amd.get_triton_quant
        xq, xs = quant(aiter_amd.QuantType.per_1x32)(st["x"], shuffle=True)
        if st["bias"] is None:
            return aiter_amd.gemm_a4w4(xq, st["w"], xs, st["w_scale"])
        return aiter_amd.gemm_a4w4(xq, st["w"], xs, st["w_scale"], bias=st["bias"], beta=1.0)
    if kind == "mxfp8":
        return aiter_amd.gemm_a8w4_mxfp8_dynamic(st["x"], st["w"], st["w_scale"])
    if kind == "bf16":
        return aiter_amd.tgemm.mm(st["x"], st["w"], st["bias"],
                                  otype=torch.float32 if case["out"] == "f32" else torch.bfloat16)
    if kind == "norm":
        (xq, xs), _, _, residual = aiter_amd.fused_rms_mxfp4_quant(st["x"], st["gamma"], EPS, res1=st["residual"],
                                                                  shuffle=True)
        return aiter_amd.gemm_a4w4(xq, st["w"], xs, st["w_scale"]), residual
    if kind == "batched":
        return aiter_amd.batched_gemm_bf16_CK(st["x"], st["w"], st["bias"])
    act = aiter_amd.ActivationType.Gelu if case["act"] == "gelu" else aiter_amd.ActivationType.Silu
    return aiter_amd.fused_moe(st["x"], st["w1"], st["w2"], st["topk_weight"], st["topk_ids"], activation=act,
                               quant_type=aiter_amd.QuantType.per_1x32, w1_scale=st["w1_scale"],
                               w2_scale=st["w2_scale"])


def work(case):
    kind, m = case["kind"], case["m"]
    if kind == "moe":
        e, topk, dim, inter = case["experts"], case["topk"], case["dim"], case["inter"]
        touched = e * (1 - (1 - topk / e) ** m)          # experts that some token goes to
        weights = touched * 3 * inter * dim * (1 / 2 + 1 / 32)
        return {"bytes": weights + 2 * 2 * m * dim + 8 * m * topk, "flops": 2 * 3 * m * topk * inter * dim}
    n, k = case["n"], case["k"]
    if kind == "batched":
        return {"bytes": 2 * case["b"] * (m * k + n * k + m * n), "flops": 2 * case["b"] * m * n * k}
    if kind == "bf16":
        return {"bytes": 2 * (m * k + n * k) + (4 if case["out"] == "f32" else 2) * m * n, "flops": 2 * m * n * k}
    rows = 2 * m * k if kind != "norm" else 3 * 2 * m * k
    return {"bytes": rows + n * k * (1 / 2 + 1 / 32) + 2 * m * n, "flops": 2 * m * n * k}


def tolerance(case):
    if case["kind"] == "bf16" and case["out"] == "f32":
        return {"rel": 1e-5, "max": 1e-4}        # f32 sums in another order
    if case["kind"] == "moe":
        # bf16 rows per routed pair and a requantised hidden row
        return {"rel": 1.2e-2, "max": 0.15}
    if case["kind"] == "norm":
        # a normalised value next to a rounding boundary moves by one e2m1 step
        return {"rel": 8e-3, "max": 0.1}
    return {"rel": 4e-3, "max": 2e-2}            # one rounding to bf16


# ------------------------------------------------------------- exact results
def _exponent_byte(amax, how, fp8):
    """e8m0 byte of a block: "even" rounds the largest magnitude to the
    nearest power of two (fp4 grid), "up" takes the power of two that holds
    amax / (largest value of the element type)."""
    bits = amax.view(torch.int32)
    if how == "even":
        return ((((bits + 0x200000) >> 23) & 0xFF) - (8 if fp8 else 2)).clamp(min=0)
    bits = (amax.clamp(min=1e-10) * (torch.ones((), device=amax.device) / (448.0 if fp8 else 6.0))).view(torch.int32)
    return (bits >> 23) + ((bits & 0x7FFFFF) != 0)


def _mx(x, how, fp8=False):
    """x [R, C] f32 -> the values its MX form stands for, in 64 bits."""
    g = x.view(x.shape[0], -1, 32)
    byte = _exponent_byte(g.abs().amax(-1), how, fp8)
    scale = torch.ldexp(torch.ones((), dtype=torch.float64, device=x.device), byte - 127)[..., None]
    v = g.double() / scale
    if fp8:
        q = v.clamp(-448, 448).float().to(torch.float8_e4m3fn).double()
    else:
        mag = v.abs().clamp(max=6.0)
        step = torch.where(mag < 2, 0.5, torch.where(mag < 4, 1.0, 2.0))
        q = torch.copysign(torch.round(mag / step) * step, v)
    return (q * scale).view(x.shape)


def _chunked(rows, w, how=None):
    """rows (64 bits) @ w^T, w in bf16, quantised per ``how`` a few thousand
    rows at a time."""
    step = max(16, (1 << 26) // w.shape[1])
    parts = [w[i:i + step].float() for i in range(0, w.shape[0], step)]
    return torch.cat([rows @ (p.double() if how is None else _mx(p, how)).t() for p in parts], 1)


def _exact_moe(case, seed):
    e, dim, inter = case["experts"], case["dim"], case["inter"]
    w1 = _weights(seed, (e * 2 * inter, dim), 1).view(e, 2 * inter, dim)
    w2 = _weights(seed, (e * dim, inter), 2).view(e, dim, inter)
    weight, ids = _routing(case, seed)
    x = _mx(_activations(seed, (case["m"], dim)).float(), "up")
    out = torch.zeros(case["m"], dim, dtype=torch.float64, device="cuda")
    for i in torch.unique(ids).tolist():
        token, slot = (ids == i).nonzero(as_tuple=True)
        h = x[token] @ _mx(w1[i].float(), "even").t()
        gate, up = h[:, :inter], h[:, inter:]
        gate = torch.nn.functional.gelu(gate) if case["act"] == "gelu" else torch.nn.functional.silu(gate)
        # the hidden rows are bf16 before they are quantised again
        h = _mx((gate * up).to(torch.bfloat16).float(), "up")
        out.index_add_(0, token, (h @ _mx(w2[i].float(), "even").t()) * weight[token, slot].double()[:, None])
    return out


def exact(case, seed):
    """What ``run`` returns, in 64 bits, with the quantisation that the entry
    points define (it is part of the result) but no other rounding."""
    kind = case["kind"]
    if kind == "moe":
        return _exact_moe(case, seed)
    if kind == "batched":
        x, w = _activations(seed, (case["b"], case["m"], case["k"])), _weights(seed, (case["b"], case["n"], case["k"]))
        y = torch.stack([x[i].double() @ w[i].double().t() for i in range(case["b"])])
        return y + _vector(seed, case["n"], 2).double() if case["bias"] else y
    x, w = _activations(seed, (case["m"], case["k"])), _weights(seed, (case["n"], case["k"]))
    if kind == "bf16":
        y = _chunked(x.double(), w)
    elif kind == "mxfp8":
        y = _chunked(_mx(x.float(), "even", True), w, "even")
    elif kind == "mxfp4":
        y = _chunked(_mx(x.float(), case["round"]), w, "even")
    else:
        r = x.double() + _activations(seed, (case["m"], case["k"]), 4).double()
        gamma = (1 + 0.1 * _vector(seed, case["k"], 5)).to(torch.bfloat16).double()
        normed = r * torch.rsqrt((r * r).mean(-1, keepdim=True) + EPS) * gamma
        return _chunked(_mx(normed.float(), "even"), w, "even"), r
    return y + _vector(seed, case["n"], 2).double() if case.get("bias") else y
