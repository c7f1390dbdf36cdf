"""Performance cases of the MXFP4 codec: what a training or serving program has it do.

Every case is one call (or one send + receive pair) of the Python entry points that
Transformer Engine's and Megatron's patches import, on device tensors. Inputs have the
distributions of the benchmark configurations: N(0, 1) activations with a few channels a
hundred times larger, and 0.02 * N(0, 1) weights with 1% heavy-tailed entries.

Results are bytes (codes, E8M0 scales, E4M3 values) or the one correctly rounded value of a
product (bf16 / fp32), so every tolerance is "exact". ``exact`` restates the floating outputs
in 64 bits with plain torch.
"""
import math
import os
import random
import sys

import numpy as np
import torch

# the packages live in a folder of the repository's root, which is the working folder
sys.path.insert(0, os.path.join(os.getcwd(), "mxfp4-hopper_amd"))

from omo_python_api import ep_payload as ep  # noqa: E402
from omo_python_api.mxfp4 import (  # noqa: E402
    omo_per_token_group_quant_mxfp4,
    omo_per_token_group_quant_mxfp4_dual,
    omo_per_token_group_quant_mxfp4_dual_grouped,
)
from omo_python_api.mxfp4_dequant import (  # noqa: E402
    omo_per_token_mxfp4RowToBf16ToFp8Col_msplit_wrapper,
    omo_per_token_mxfp4RowToBf16ToFp8Col_wrapper,
    omo_per_token_mxfp4ToBf16_dequant_wrapper,
    omo_per_token_mxfp4ToFp8_wrapper,
)
from omo_python_api.mxfp4_tensor import MXFP4Quantizer  # noqa: E402
from omo_python_api.permutation import mxfp4_permute_to_fp8  # noqa: E402

EPS = 1e-10
E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)
LARGEST = 7168 * 2048 * 24  # elements of the largest listed case


# ------------------------------------------------------------------------------ the cases
def listed():
    return [
        # One decode step's activations of 16 sequences, quantized for an MXFP4 linear
        # layer: the smallest call, launch latency and host time.
        {"name": "quantize_decode", "kind": "quantize", "rows": 16, "cols": 7168},
        # A prefill or training batch's activations, rowwise: the headline workload.
        {"name": "quantize_prefill", "kind": "quantize", "rows": 8192, "cols": 7168},
        # A dense FFN weight in both layouts, once per optimizer step.
        {"name": "quantize_weight", "kind": "dual", "rows": 7168, "cols": 18432},
        # All local experts' weights (gate + up fused, and down) of one MoE layer in
        # both layouts, in one call: the largest.
        {"name": "quantize_experts", "kind": "dual_grouped", "count": 8, "hidden": 7168, "ffn": 2048},
        # MXFP4 activations back to bf16 for an operation without an FP4 path.
        {"name": "dequantize_bf16", "kind": "dequantize", "rows": 8192, "cols": 7168, "dtype": "bfloat16"},
        # An expert weight held as an MXFP4Tensor to fp32, as optimizers and checkpoints
        # take it (float32 is the tensor class's default).
        {"name": "dequantize_fp32", "kind": "dequantize", "rows": 7168, "cols": 2048, "dtype": "float32"},
        # Forward GEMM input of 8 local experts: MXFP4 to FP8 with 1x128 scales, split per expert.
        {"name": "requant_experts", "kind": "requant", "rows": 4096, "cols": 7168, "splits": 8},
        # The same for a dense layer whose width is not a multiple of 128 (the wrapper pads it).
        {"name": "requant_padded", "kind": "requant", "rows": 4096, "cols": 2880, "splits": 1},
        # Backward (wgrad) input of a dense layer: rowwise MXFP4 to columnwise FP8.
        {"name": "wgrad_dense", "kind": "wgrad", "rows": 4096, "cols": 7168},
        # Backward (wgrad) input of 8 local experts with ragged row counts.
        {"name": "wgrad_experts", "kind": "wgrad_splits", "rows": 16431, "cols": 7168, "splits": 8},
        # Expert-parallel exchange of one GPU's tokens: quantize into payload rows
        # (send), FP8 from payload rows per expert (receive).
        {"name": "payload_exchange", "kind": "payload", "rows": 4096, "cols": 7168, "splits": 8},
        # Top-8 of 64 routing of MXFP4 tokens into expert-major FP8 rows.
        {"name": "permute_experts", "kind": "permute", "rows": 4096, "cols": 7168, "experts": 64, "topk": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _multiple(rng, lo, hi, m):
    return min(hi // m * m, max(m, (_log_int(rng, lo, hi) + m // 2) // m * m))


def draw(rng):
    """One more case: any kind, sizes over the whole range (decode batches to prefill
    batches; widths from 1024 up), ragged row counts and widths that are not multiples of
    the tiles among them."""
    kind = rng.choice(["quantize", "dual", "dual_grouped", "dequantize", "requant", "wgrad", "wgrad_splits", "payload",
                       "permute"])
    if kind == "quantize":
        return {"kind": kind, "rows": _log_int(rng, 1, 16431), "cols": _multiple(rng, 1024, 18432, 32)}
    if kind == "dual":
        return {"kind": kind, "rows": _multiple(rng, 32, 16384, 32), "cols": _multiple(rng, 1024, 18432, 32)}
    if kind == "dual_grouped":
        return {"kind": kind, "count": rng.randint(1, 8), "hidden": _multiple(rng, 1024, 7168, 32),
                "ffn": _multiple(rng, 256, 2048, 32)}
    if kind == "dequantize":  # the entry point takes multiples of 128 code bytes
        return {"kind": kind, "rows": _multiple(rng, 4, 8192, 4), "cols": _multiple(rng, 1024, 7168, 64),
                "dtype": rng.choice(["bfloat16", "float32"])}
    if kind == "requant":  # the entry point takes multiples of 128 (padded) code bytes
        return {"kind": kind, "rows": _multiple(rng, 2, 16384, 2), "cols": _multiple(rng, 1024, 7168, 32),
                "splits": rng.choice([1, 2, 4, 8, 16, 32])}
    if kind == "wgrad":
        return {"kind": kind, "rows": _log_int(rng, 32, 16384), "cols": _multiple(rng, 1024, 7168, 32)}
    if kind == "wgrad_splits":
        return {"kind": kind, "rows": _log_int(rng, 256, 16431), "cols": _multiple(rng, 1024, 7168, 32),
                "splits": rng.choice([2, 4, 8, 16, 32])}
    if kind == "payload":
        return {"kind": kind, "rows": _log_int(rng, 1, 8192), "cols": _multiple(rng, 1024, 7168, 128),
                "splits": rng.choice([1, 2, 4, 8, 16])}
    experts = rng.choice([8, 16, 32, 64])
    return {"kind": kind, "rows": _log_int(rng, 16, 4096), "cols": _multiple(rng, 1024, 7168, 128),
            "experts": experts, "topk": rng.randint(1, 8)}


def _splits(rows, n):
    """Uneven expert loads that sum to ``rows``, fixed by the case."""
    r = random.Random(rows * 1009 + n)
    w = [r.uniform(0.5, 1.5) for _ in range(n)]
    cuts = [round(rows * sum(w[:i]) / sum(w)) for i in range(n + 1)]
    return [b - a for a, b in zip(cuts, cuts[1:])]


def _expert_shapes(case):
    """fc1 (gate + up) and fc2 weights, [out, in], of every local expert."""
    h, f = case["hidden"], case["ffn"]
    return [(2 * f, h)] * case["count"] + [(h, f)] * case["count"]


# ----------------------------------------------------------------------------- the inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _activations(rows, cols, g):
    x = torch.randn((rows, cols), generator=g, device="cuda")
    x[:, torch.randperm(cols, generator=g, device="cuda")[:max(1, round(0.001 * cols))]] *= 100.0
    return x.to(torch.bfloat16)


def _weights(rows, cols, g):
    w = torch.randn((rows, cols), generator=g, device="cuda")
    k = rows * cols // 100
    pos = torch.randperm(rows * cols, generator=g, device="cuda")[:k]
    chi = torch.randn((k, 3), generator=g, device="cuda").square().sum(1)
    w.view(-1)[pos] = torch.randn((k,), generator=g, device="cuda") / torch.sqrt(chi / 3.0)  # Student-t(3)
    return (w * 0.02).to(torch.bfloat16)


def _encode(x):
    """MXFP4 codes and E8M0 scale bytes of a [M, K] bf16 tensor, in plain torch."""
    M, K = x.shape
    b = x.float().view(M, K // 32, 32)
    m, e = torch.frexp(b.abs().amax(-1).clamp_min(EPS))  # amax = m * 2^e, m in [0.5, 1)
    k = e - 3 + (m > 0.75).int()                          # ceil(log2(amax / 6))
    v = torch.ldexp(b, -k.unsqueeze(-1))
    a = v.abs()
    code = (a > 0.25).to(torch.uint8)
    for above in (a >= 0.75, a > 1.25, a >= 1.75, a > 2.5, a >= 3.5, a > 5.0):  # ties to even
        code += above
    code |= torch.signbit(v).to(torch.uint8) << 3
    code = code.view(M, K)
    return code[:, 0::2] | (code[:, 1::2] << 4), (k + 127).to(torch.uint8)


def _routing(tokens, experts, topk, g):
    """Boolean routing map [tokens, experts], topk distinct experts per token."""
    choice = torch.rand((tokens, experts), generator=g, device="cuda").topk(topk, dim=1).indices
    return torch.zeros((tokens, experts), dtype=torch.bool, device="cuda").scatter_(1, choice, True)


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    state = {"kind": kind}
    if kind == "quantize":
        state["x"] = _activations(case["rows"], case["cols"], g)
    elif kind == "dual":
        state["x"] = _weights(case["rows"], case["cols"], g)
    elif kind == "dual_grouped":
        state["xs"] = [_weights(m, k, g) for m, k in _expert_shapes(case)]
    elif kind == "payload":
        state["x"] = _activations(case["rows"], case["cols"], g)
        state["splits"] = _splits(case["rows"], case["splits"])
    elif kind == "dequantize" and case["dtype"] == "float32":
        state["kind"] = "dequantize_tensor"
        state["tensor"] = MXFP4Quantizer(rowwise=True, columnwise=False)(_weights(case["rows"], case["cols"], g))
        state["dtype"] = torch.float32
    else:
        state["codes"], state["scales"] = _encode(_activations(case["rows"], case["cols"], g))
        if kind == "dequantize":
            state["dtype"] = getattr(torch, case["dtype"])
        if kind in ("requant", "wgrad_splits"):
            state["splits"] = _splits(case["rows"], case["splits"])
        if kind == "permute":
            state["routing"] = _routing(case["rows"], case["experts"], case["topk"], g)
    return state


# --------------------------------------------------------------------------------- a pass
def run(state):
    kind = state["kind"]
    if kind == "quantize":
        return omo_per_token_group_quant_mxfp4(state["x"])
    if kind == "dual":
        return omo_per_token_group_quant_mxfp4_dual(state["x"])
    if kind == "dual_grouped":
        return omo_per_token_group_quant_mxfp4_dual_grouped(state["xs"])
    if kind == "dequantize":
        return omo_per_token_mxfp4ToBf16_dequant_wrapper(state["codes"], state["scales"], state["dtype"])
    if kind == "dequantize_tensor":
        return state["tensor"].dequantize(dtype=state["dtype"])
    if kind == "requant":
        return omo_per_token_mxfp4ToFp8_wrapper(state["codes"], state["scales"], state["splits"])
    if kind == "wgrad":
        return omo_per_token_mxfp4RowToBf16ToFp8Col_wrapper(state["codes"], state["scales"])
    if kind == "wgrad_splits":
        return omo_per_token_mxfp4RowToBf16ToFp8Col_msplit_wrapper(state["codes"], state["scales"], state["splits"])
    if kind == "payload":
        payload = ep.fp4_quantize_packed(state["x"])
        return payload, ep.packed_mxfp4ToFp8(payload, state["splits"])
    x_q, x_s, src, m_splits = mxfp4_permute_to_fp8(state["codes"], state["scales"], state["routing"], split=False)
    return x_q, x_s, src, np.array(m_splits)


# -------------------------------------------------------------------- what a pass cannot do without
def _ceil(a, b):
    return -(-a // b)


def work(case):
    kind = case["kind"]
    if kind == "dual_grouped":
        n = sum(m * k for m, k in _expert_shapes(case))
        return {"bytes": 2 * n + 2 * (n // 2 + n // 32), "flops": 0}
    M, K = case["rows"], case["cols"]
    n, mx = M * K, M * K // 2 + M * K // 32  # elements; MXFP4 bytes
    fp8 = n + 4 * M * _ceil(K, 128)          # E4M3 values and 1x128 scales
    if kind == "quantize":
        b = 2 * n + mx
    elif kind == "dual":
        b = 2 * n + 2 * mx
    elif kind == "dequantize":
        b = mx + n * (4 if case["dtype"] == "float32" else 2)
    elif kind == "requant":
        b = mx + fp8
    elif kind == "wgrad":
        b = mx + n + 4 * K * _ceil(M, 128)
    elif kind == "wgrad_splits":
        b = mx + n + 4 * K * sum(_ceil(m, 128) for m in _splits(M, case["splits"]))
    elif kind == "payload":
        b = 2 * n + 2 * mx + fp8
    else:
        b = mx + M * case["experts"] + case["topk"] * (fp8 + 4 * M)
    return {"bytes": b, "flops": 0}


def tolerance(case):
    return "exact"  # bytes, correctly rounded products and powers of two: nothing is summed


# ------------------------------------------------------------------------------ in 64 bits
def _decode(codes, scales):
    """The signed E2M1 values [M, K] of the codes and the block scales' exponents [M, K], in float64."""
    M, K = codes.shape[0], codes.shape[1] * 2
    c = torch.stack((codes & 15, codes >> 4), -1).view(M, K).long()
    t = torch.tensor(E2M1 + tuple(-v for v in E2M1), dtype=torch.float64, device=codes.device)
    return t[c], (scales.double() - 127.0).repeat_interleave(32, dim=1)


def _requant64(codes, scales):
    """FP8 values before rounding and 1x128 scales: the group's scale is the largest
    block scale / 64; a zero of a block 2^7 or more below it reads as -448 (+448 for -0),
    which is how the format's consumer defines it."""
    v, e = _decode(codes, scales)
    M, K = v.shape
    negative_zero = torch.stack((codes & 15, codes >> 4), -1).view(M, K) == 8
    P = _ceil(K, 128) * 128
    top = torch.nn.functional.pad(e, (0, P - K), value=-127.0).view(M, P // 128, 128).amax(-1)
    d = top.repeat_interleave(128, dim=1)[:, :K] - 6.0 - e
    q = torch.clamp(v * torch.exp2(-d), -448.0, 448.0)
    wrapped = torch.where(negative_zero, 448.0, -448.0).double()
    return torch.where((v == 0) & (d >= 1), wrapped, q), torch.exp2(top - 6.0).t()


def _column64(v, pow2):
    """One split's FP8 columns [K, m] before rounding and their scales [ceil(m / 128), K]."""
    m, K = v.shape
    T = _ceil(m, 128)
    amax = torch.nn.functional.pad(v.abs(), (0, 0, 0, T * 128 - m)).view(T, 128, K).amax(1)
    if pow2:
        s = torch.where(amax <= EPS, torch.ones_like(amax), torch.exp2(torch.ceil(torch.log2(amax / 448.0))))
    else:
        s = amax.clamp_min(EPS) / 448.0
    return (v / s.repeat_interleave(128, dim=0)[:m]).t(), s


def exact(case, seed):
    """The floating outputs in 64 bits; None in the place of bytes (codes, scale bytes,
    row numbers), which have no value closer to the truth than their own."""
    kind = case["kind"]
    if kind in ("quantize", "dual", "dual_grouped"):
        return None
    if kind == "payload":
        codes, scales = _encode(prepare(case, seed)["x"])
    elif kind == "dequantize" and case["dtype"] == "float32":
        codes, scales = _encode(_weights(case["rows"], case["cols"], _gen(seed)))
    else:
        state = prepare(case, seed)
        codes, scales = state["codes"], state["scales"]
    if kind == "dequantize":
        v, e = _decode(codes, scales)
        return v * torch.exp2(e)
    if kind in ("wgrad", "wgrad_splits"):
        v, e = _decode(codes, scales)
        v = v * torch.exp2(e)
        if kind == "wgrad":
            return _column64(v, False)
        parts = [_column64(p, True) for p in torch.split(v, state["splits"])]
        return [p[0] for p in parts], [p[1] for p in parts]
    if kind == "permute":
        src = torch.nonzero(state["routing"].t(), as_tuple=True)[1]
        q, s = _requant64(codes, scales)
        return q[src], s[:, src], None, None
    q, s = _requant64(codes, scales)
    lens = _splits(case["rows"], case["splits"])
    pair = (torch.split(q, lens, dim=0), torch.split(s, lens, dim=1))
    return (None, pair) if kind == "payload" else pair
