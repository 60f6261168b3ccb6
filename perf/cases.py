"""Timed cases of the block-FP8 path: its public calls over the sizes, types and options that a
program using it has.

A case is a dict of plain values with a "kind" (the call) and its sizes:

  gemm    w8a8_block_fp8_matmul on operands quantised before: the matmul alone (M, N, K, out)
  linear  bf16 activations through a quantised linear layer (M, N, K, out): the in-op quantiser
          (act_quant_w8a8_block_fp8_matmul) where the layer's input width is whole groups of
          128, else act_quant followed by w8a8_block_fp8_matmul
  rows    gemm_fp8_fp8_bf16_nt: one weight scale per row and 128 columns (M, N, K)
  quant   act_quant of activations (M, K, dtype, group)
  silu    silu_and_mul_quant, the quantising half of a gated MLP (M, K = the gate's width)
  weight  quantize_weight, the offline 128x128 quantiser (N, K, dtype)
  mlp     fp8_mlp, the whole gated MLP (M, H, I), gate/up interleaved or not

Activations are N(0, 1) in bf16, with 1% of the values times 20 where "outliers" is set (the
range that makes per-group scales worth having); weights are N(0, 0.02) with one scale per
128x128 block.
"""
from __future__ import annotations

import math

import torch

from hf_kernels_helion_amd import deep_gemm_helion, finegrained_fp8_helion as fp8

FP8 = torch.float8_e4m3fn
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZEOF = {"bf16": 2, "fp16": 2, "fp32": 4}


def listed():
    return [
        # A small projection: latency and launches, not the matrix cores.
        {"name": "gemm_small", "kind": "gemm", "M": 512, "N": 512, "K": 2048, "out": "bf16"},
        # A mid-size layer on outlier-heavy activations.
        {"name": "gemm_mid", "kind": "gemm", "M": 2048, "N": 2048, "K": 4096, "out": "bf16",
         "outliers": True},
        # The compute-bound prefill GEMM.
        {"name": "gemm_large", "kind": "gemm", "M": 4096, "N": 4096, "K": 8192, "out": "bf16"},
        # A prefill chunk with the matmul's default output type.
        {"name": "gemm_fp32_out", "kind": "gemm", "M": 1000, "N": 4096, "K": 7168, "out": "fp32"},
        # A decode batch through a down projection, activations quantised in the op.
        {"name": "linear_decode_32", "kind": "linear", "M": 32, "N": 4096, "K": 14336,
         "out": "bf16"},
        # One token through a gate/up projection.
        {"name": "linear_decode_1", "kind": "linear", "M": 1, "N": 28672, "K": 4096,
         "out": "bf16"},
        # An eighth of an 11008-wide intermediate layer: 10.75 groups of 128.
        {"name": "linear_ragged", "kind": "linear", "M": 777, "N": 4096, "K": 1376,
         "out": "bf16"},
        # The per-row-scale matmul at prefill size.
        {"name": "rows_prefill", "kind": "rows", "M": 4096, "N": 4096, "K": 8192},
        # Prefill activations on their own.
        {"name": "quant_prefill", "kind": "quant", "M": 4096, "K": 8192, "dtype": "bf16",
         "group": 128, "outliers": True},
        # One weight of a checkpoint being quantised.
        {"name": "weight_bf16", "kind": "weight", "N": 4096, "K": 14336, "dtype": "bf16"},
        # A whole gated MLP: a prompt with a ragged token count, and a decode batch.
        {"name": "mlp_prefill", "kind": "mlp", "M": 3001, "H": 4096, "I": 14336,
         "interleaved": True},
        {"name": "mlp_decode", "kind": "mlp", "M": 8, "H": 4096, "I": 14336,
         "interleaved": False},
    ]


def _spread(rng, lo, hi, step=1):
    """A size between lo and hi, even over its logarithm, a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choices(["gemm", "linear", "ragged", "rows", "quant", "silu", "weight", "mlp"],
                       [6, 6, 3, 3, 3, 2, 2, 4])[0]
    # layer widths: whole 128-blocks mostly, else any multiple of 8
    width = 128 if rng.random() < 0.8 else 8
    if kind in ("gemm", "linear", "rows"):
        # decode batches up to prefill chunks; K in whole groups
        while True:
            c = {"kind": kind, "M": _spread(rng, 1, 8192), "N": _spread(rng, 512, 28672, width),
                 "K": _spread(rng, 512, 14336, 128)}
            if c["M"] * c["N"] * c["K"] <= 4096 * 4096 * 8192:
                break
        if kind != "rows":
            c["out"] = rng.choices(["bf16", "fp32", "fp16"], [6, 3, 1])[0]
            c["outliers"] = rng.random() < 0.3
        return c
    if kind == "ragged":
        # input widths that are not whole groups of 128 (shards of odd intermediate sizes),
        # most of them multiples of 16 or 8
        while True:
            c = {"kind": "linear", "M": _spread(rng, 1, 4096), "N": _spread(rng, 256, 8192, width),
                 "K": _spread(rng, 256, 5504, rng.choices([16, 8, 1], [5, 2, 1])[0]),
                 "out": rng.choices(["bf16", "fp32"], [3, 1])[0]}
            if c["K"] % 128 and c["M"] * c["N"] * c["K"] <= 777 * 4096 * 1376:
                return c
    if kind == "quant":
        while True:
            c = {"kind": "quant", "M": _spread(rng, 1, 16384),
                 "K": _spread(rng, 512, 16384, rng.choices([128, 8], [4, 1])[0]),
                 "dtype": rng.choices(["bf16", "fp16", "fp32"], [4, 1, 1])[0],
                 "group": rng.choices([128, 64], [5, 1])[0], "outliers": rng.random() < 0.5}
            if c["M"] * c["K"] <= 2 * 4096 * 8192:
                return c
    if kind == "silu":
        return {"kind": "silu", "M": _spread(rng, 1, 3001), "K": _spread(rng, 512, 14336, 128)}
    if kind == "weight":
        return {"kind": "weight", "N": _spread(rng, 256, 14336, width),
                "K": _spread(rng, 512, 14336, width), "dtype": rng.choice(["bf16", "fp32"])}
    while True:
        c = {"kind": "mlp", "M": _spread(rng, 1, 4096), "H": _spread(rng, 1024, 8192, 128),
             "I": _spread(rng, 1024, 14336, 128), "interleaved": rng.random() < 0.5}
        if c["M"] * c["H"] * c["I"] <= 3001 * 4096 * 14336:
            return c


# ------------------------------------------------------------------ inputs


def _activations(g, M, K, dtype, outliers):
    x = torch.randn(M, K, generator=g, device="cuda")
    if outliers:
        x *= 1.0 + 19.0 * (torch.rand(M, K, generator=g, device="cuda") < 0.01)
    return x.to(dtype)


def _scales(amax):
    # (by a tensor: a division by a number is a product with its rounded reciprocal on the GPU)
    return amax.clamp_min(1e-10) / torch.full_like(amax, 448.0)


def _act_quant(x, group=128):
    """Codes and scales of the activation quantiser's contract, in plain torch."""
    M, K = x.shape
    G = -(-K // group)
    v = torch.nn.functional.pad(x.float(), (0, G * group - K)).view(M, G, group)
    s = _scales(v.abs().amax(dim=2))
    q = (v / s[:, :, None]).to(FP8).view(M, G * group)[:, :K].contiguous()
    return q, s


def _weight_quant(W, bn=128):
    """Codes and scales per bn x 128 block, in plain torch."""
    N, K = W.shape
    NB, KB = -(-N // bn), -(-K // 128)
    v = torch.nn.functional.pad(W.float(), (0, KB * 128 - K, 0, NB * bn - N))
    v = v.view(NB, bn, KB, 128)
    s = _scales(v.abs().amax(dim=(1, 3)))
    q = (v / s[:, None, :, None]).to(FP8).view(NB * bn, KB * 128)[:N, :K].contiguous()
    return q, s


def _weight(g, N, K, bn=128):
    return _weight_quant(0.02 * torch.randn(N, K, generator=g, device="cuda"), bn)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind, outliers = case["kind"], case.get("outliers", False)
    st = {"case": dict(case)}
    if kind in ("gemm", "rows"):
        st["A"], st["As"] = _act_quant(_activations(g, case["M"], case["K"], torch.bfloat16,
                                                    outliers))
        st["B"], st["Bs"] = _weight(g, case["N"], case["K"], 1 if kind == "rows" else 128)
    elif kind == "linear":
        st["x"] = _activations(g, case["M"], case["K"], torch.bfloat16, outliers)
        st["B"], st["Bs"] = _weight(g, case["N"], case["K"])
    elif kind == "quant":
        st["x"] = _activations(g, case["M"], case["K"], DTYPES[case["dtype"]], outliers)
    elif kind == "silu":
        st["x"] = _activations(g, case["M"], 2 * case["K"], torch.bfloat16, False)
    elif kind == "weight":
        W = 0.02 * torch.randn(case["N"], case["K"], generator=g, device="cuda")
        st["W"] = W.to(DTYPES[case["dtype"]])
    else:
        M, H, I = case["M"], case["H"], case["I"]
        st["x"] = _activations(g, M, H, torch.bfloat16, False)
        w, s = _weight(g, 2 * I, H)
        st["wd"], st["sd"] = _weight(g, H, I)
        st["wg"], st["sg"] = fp8.interleave_gate_up(w, s) if case["interleaved"] else (w, s)
    return st


# ------------------------------------------------------------------ the calls


def run(st):
    c = st["case"]
    kind = c["kind"]
    if kind == "gemm":
        return fp8.w8a8_block_fp8_matmul(st["A"], st["B"], st["As"], st["Bs"], [128, 128],
                                         DTYPES[c["out"]])
    if kind == "linear":
        out = DTYPES[c["out"]]
        if c["K"] % 128 == 0:
            return fp8.act_quant_w8a8_block_fp8_matmul(st["x"], st["B"], st["Bs"], [128, 128], out)
        q, s = fp8.act_quant(st["x"], 128)
        return fp8.w8a8_block_fp8_matmul(q, st["B"], s, st["Bs"], [128, 128], out)
    if kind == "rows":
        return deep_gemm_helion.gemm_fp8_fp8_bf16_nt(st["A"], st["B"], st["As"], st["Bs"])
    if kind == "quant":
        return fp8.act_quant(st["x"], c["group"])
    if kind == "silu":
        return fp8.silu_and_mul_quant(st["x"], 128)
    if kind == "weight":
        return fp8.quantize_weight(st["W"])
    return fp8.fp8_mlp(st["x"], st["wg"], st["sg"], st["wd"], st["sd"],
                       gate_up_interleaved=c["interleaved"])


def work(case):
    kind = case["kind"]
    up = lambda n: -(-n // 128)  # noqa: E731
    if kind in ("gemm", "linear", "rows"):
        M, N, K = case["M"], case["N"], case["K"]
        a = 2 * M * K if kind == "linear" else M * K + 4 * M * up(K)
        b = N * K + 4 * (N if kind == "rows" else up(N)) * up(K)
        return {"bytes": a + b + M * N * SIZEOF[case.get("out", "bf16")], "flops": 2 * M * N * K}
    if kind == "quant":
        M, K = case["M"], case["K"]
        return {"bytes": M * K * (SIZEOF[case["dtype"]] + 1) + 4 * M * -(-K // case["group"]),
                "flops": 3 * M * K}
    if kind == "silu":
        M, K = case["M"], case["K"]
        return {"bytes": M * K * 5 + 4 * M * up(K), "flops": 10 * M * K}
    if kind == "weight":
        N, K = case["N"], case["K"]
        return {"bytes": N * K * (SIZEOF[case["dtype"]] + 1) + 4 * up(N) * up(K),
                "flops": 3 * N * K}
    M, H, I = case["M"], case["H"], case["I"]
    return {"bytes": 4 * M * H + 3 * I * H + 12 * up(I) * up(H), "flops": 6 * M * H * I}


def tolerance(case):
    kind = case["kind"]
    if kind in ("quant", "weight"):
        return "exact"  # codes and scales are defined bit for bit
    if kind == "silu":
        # silu in fp32 rounded twice to bf16, then codes of 3 mantissa bits: an ulp of the
        # first moves a code now and then
        return {"rel": 5e-3, "max": 0.15}
    if kind == "mlp":
        # two bf16 roundings and a requantisation between the matmuls
        return {"rel": 8e-3, "max": 0.05}
    # One rounding of the result (2^-9 relative in bf16, 2^-12 in fp16), or the fp32 sums of
    # 128-long fp8 products. Measured against 64 bits: 1.7e-3, 2.1e-4 and 1.4e-5.
    return {"bf16": {"rel": 7e-3, "max": 2e-2}, "fp16": {"rel": 8e-4, "max": 4e-3},
            "fp32": {"rel": 6e-5, "max": 1e-3}}[case.get("out", "bf16")]


# ------------------------------------------------------------------ the same in 64 bits


def _deq(q, s, bn):
    """Codes times their block scales (bn rows by 128 columns) in float64."""
    e = s.double().repeat_interleave(bn, 0)[:q.shape[0]]
    return q.double() * e.repeat_interleave(128, 1)[:, :q.shape[1]]


def _matmul(q, s, B, Bs, bn=128):
    return _deq(q, s, 1) @ _deq(B, Bs, bn).t()


def exact(case, seed):
    st = prepare(case, seed)
    kind = case["kind"]
    if kind in ("gemm", "rows"):
        return _matmul(st["A"], st["As"], st["B"], st["Bs"], 1 if kind == "rows" else 128)
    if kind == "linear":
        q, s = _act_quant(st["x"])  # the codes are the contract; the products are exact
        return _matmul(q, s, st["B"], st["Bs"])
    if kind == "quant":
        M, K, group = case["M"], case["K"], case["group"]
        x = st["x"].double()
        G = -(-K // group)
        v = torch.nn.functional.pad(x, (0, G * group - K)).view(M, G, group)
        s = v.abs().amax(dim=2).clamp_min(1e-10) / 448.0
        return (v / s[:, :, None]).view(M, G * group)[:, :K].contiguous(), s
    if kind == "silu":
        d = case["K"]
        a, b = st["x"][:, :d].double(), st["x"][:, d:].double()
        v = (a * torch.sigmoid(a) * b).view(-1, d // 128, 128)
        s = v.abs().amax(dim=2).clamp_min(1e-10) / 448.0
        return (v / s[:, :, None]).view(-1, d), s
    if kind == "weight":
        N, K = st["W"].shape
        NB, KB = -(-N // 128), -(-K // 128)
        v = torch.nn.functional.pad(st["W"].double(), (0, KB * 128 - K, 0, NB * 128 - N))
        v = v.view(NB, 128, KB, 128)
        s = v.abs().amax(dim=(1, 3)).clamp_min(1e-10) / 448.0
        q = (v / s[:, None, :, None]).view(NB * 128, KB * 128)[:N, :K].contiguous()
        return q, s
    # The MLP's rounding points (bf16 gate/up, silu and product, then the codes) are its
    # contract; the matmuls and the silu are in 64 bits.
    I = case["I"]
    q, s = _act_quant(st["x"])
    h = _matmul(q, s, st["wg"], st["sg"]).to(torch.bfloat16)
    if case["interleaved"]:
        h = h.view(-1, I // 128, 2, 128).transpose(1, 2).reshape(-1, 2 * I)
    a = h[:, :I].double()
    a = (a * torch.sigmoid(a)).to(torch.bfloat16).double() * h[:, I:].double()
    q, s = _act_quant(a.to(torch.bfloat16))
    return _matmul(q, s, st["wd"], st["sd"])
