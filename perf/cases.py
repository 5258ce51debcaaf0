"""The workloads whose speed this library answers for, as a program calls them.

Each case goes through the Python entry points of ``tx`` with tensors that the
program already holds on the GPU.  Sizes are those of this repository's own
configurations, tests and benchmark (the reference's matmul sizes 256 .. 4096,
linear layers of 4096 x 14336, 64 experts of 2048 x 4096, 16 Mi converted
values, 64 Mi scattered updates), and ``draw`` spreads each family over its
whole range, odd sizes included.

Inputs follow the repository's workload generators: uniform or normal GEMM
operands, absmax-quantised fp8 weights, Zipf(1.1) scatter keys, a skewed
expert router, converted values spread over fp8's normal and subnormal range.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "triton-ext_amd"))
import tx  # noqa: E402

DEV = "cuda"
FMAX = {torch.float8_e4m3fn: 448.0, torch.float8_e5m2: 57344.0}
DT = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16, "int32": torch.int32,
      "e4m3fn": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
SIZE = {"fp32": 4, "int32": 4, "bf16": 2, "fp16": 2, "e4m3fn": 1, "e5m2": 1}


def listed():
    return [
        # The reference's matmul(a, b): fp16, row-major b.  Its benchmark's smallest size, where
        # the call and one launch are all there is, and its largest.
        {"name": "matmul_fp16_256", "kind": "matmul", "M": 256, "N": 256, "K": 256, "dtype": "fp16", "b": "kn"},
        {"name": "matmul_fp16_4096", "kind": "matmul", "M": 4096, "N": 4096, "K": 4096, "dtype": "fp16", "b": "kn"},
        # tt.dot on odd sizes: rows off every alignment the tiles like, one column past a tile.
        {"name": "dot_bf16_ragged", "kind": "matmul", "M": 4095, "N": 4097, "K": 4100, "dtype": "bf16", "b": "nk"},
        # tt.dot with its accumulator (a K chunk added to fp32 sums: gradient accumulation, K loops).
        {"name": "dot_acc_bf16_2048", "kind": "dot_acc", "M": 2048, "N": 2048, "K": 2048, "dtype": "bf16",
         "b": "nk"},
        # fp8 linear layers as a program runs them: quantise the bf16 activations row by row, then
        # the scaled product with resident fp8 weights.  A decode batch and a prefill chunk.
        {"name": "fp8_linear_decode", "kind": "fp8_linear", "M": 16, "N": 14336, "K": 4096, "act": "none",
         "bias": False, "out": "bf16"},
        {"name": "fp8_linear_prefill", "kind": "fp8_linear", "M": 512, "N": 4096, "K": 14336, "act": "none",
         "bias": False, "out": "bf16"},
        # The fp8 product alone, operands already quantised: the largest.
        {"name": "fp8_gemm_8192", "kind": "fp8_gemm", "M": 8192, "N": 8192, "K": 8192},
        # An MX linear layer: block-quantised activations, block-scaled product.
        {"name": "mx_linear_512", "kind": "mx_linear", "M": 512, "N": 14336, "K": 4096, "fmt": "e4m3fn",
         "out": "bf16"},
        # A mixture-of-experts layer: 8192 routed rows over 64 experts, group sizes on the device.
        {"name": "moe_fp8_64x128", "kind": "moe", "G": 64, "rows": 8192, "N": 2048, "K": 4096},
        # Batch-4 decode over fp8 weights with group scales.
        {"name": "gemv_e5m2_m4", "kind": "gemv", "M": 4, "N": 14336, "K": 4096, "fmt": "e5m2"},
        # fp32 -> fp8 -> fp32, the round trip of the conversion configuration: both directions.
        {"name": "fp8_round_trip_16mi", "kind": "round_trip", "n": 1 << 24, "src": "fp32", "fmt": "e4m3fn",
         "saturate": False},
        # Scatter-reduce of Zipf keys (embedding gradients, token counts), bins zeroed first.
        {"name": "scatter_f32_64mi", "kind": "scatter", "n": 1 << 26, "nbins": 65536, "dtype": "fp32", "zipf": 1.1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dim(rng, lo, hi, step, odd=0.25):
    """A size between lo and hi, even over its logarithm; a multiple of step, or any number."""
    v = _log(rng, lo, hi)
    return v if rng.random() < odd else max(step, v // step * step)


def draw(rng):
    kind = rng.choice(["matmul", "matmul", "dot_acc", "fp8_linear", "fp8_linear", "fp8_gemm", "mx_linear",
                       "moe", "gemv", "round_trip", "scatter"])
    if kind in ("matmul", "dot_acc"):
        return {"kind": kind, "M": _dim(rng, 64, 4096, 64), "N": _dim(rng, 64, 4096, 64),
                "K": _dim(rng, 64, 4096, 64), "dtype": rng.choice(["fp16", "bf16"]), "b": rng.choice(["kn", "nk"])}
    if kind == "fp8_linear":
        return {"kind": kind, "M": _dim(rng, 1, 4096, 16, 0.4), "N": _dim(rng, 1024, 14336, 128, 0.1),
                "K": _dim(rng, 1024, 14336, 128, 0.1), "act": rng.choice(["none", "none", "relu", "gelu_tanh", "silu"]),
                "bias": rng.random() < 0.5, "out": rng.choice(["bf16", "bf16", "fp16", "fp32"])}
    if kind == "fp8_gemm":
        return {"kind": kind, "M": _dim(rng, 16, 8192, 64), "N": _dim(rng, 1024, 8192, 64),
                "K": _dim(rng, 1024, 8192, 64, 0.1)}
    if kind == "mx_linear":
        return {"kind": kind, "M": _dim(rng, 16, 4096, 32), "N": _dim(rng, 1024, 14336, 128, 0.1),
                "K": max(1, _log(rng, 1024, 8192) // 32) * 32, "fmt": rng.choice(["e4m3fn", "e4m3fn", "e5m2"]),
                "out": rng.choice(["bf16", "fp16", "fp32"])}
    if kind == "moe":
        return {"kind": kind, "G": _log(rng, 8, 128), "rows": _log(rng, 128, 8192), "N": _dim(rng, 1024, 4096, 128, 0.1),
                "K": _log(rng, 1024, 4096) // 128 * 128}
    if kind == "gemv":
        return {"kind": kind, "M": _log(rng, 1, 16), "N": _dim(rng, 1024, 14336, 64),
                "K": _log(rng, 1024, 14336) // 128 * 128, "fmt": rng.choice(["e5m2", "e4m3fn"])}
    if kind == "round_trip":
        return {"kind": kind, "n": _dim(rng, 1 << 10, 1 << 24, 256, 0.5), "src": rng.choice(["fp32", "bf16", "fp16"]),
                "fmt": rng.choice(["e4m3fn", "e5m2"]), "saturate": rng.random() < 0.5}
    return {"kind": kind, "n": _dim(rng, 1 << 16, 1 << 26, 256, 0.5), "nbins": _log(rng, 256, 1 << 20),
            "dtype": rng.choice(["fp32", "int32"]), "zipf": rng.choice([0.0, 1.1])}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _normal(g, shape, dtype=torch.float32, std=1.0):
    x = torch.empty(shape, dtype=torch.float32, device=DEV).normal_(0.0, std, generator=g)
    return x.to(dtype)


def _quant_rows(x, dtype):
    """Per-row absmax quantisation in fp32: (codes, scales) with x ~= codes * scales."""
    fmax = FMAX[dtype]
    amax = x.float().abs().amax(dim=1)
    amax = torch.where(amax > 0, amax, torch.ones_like(amax))
    top = torch.full_like(amax, fmax)
    q = (x.float() * (top / amax)[:, None]).clamp(-fmax, fmax).to(dtype)
    return q, amax / top


def _quant_blocks(x, dtype):
    """MX quantisation: one power-of-two scale (its e8m0 code) per 32 values of a row."""
    fmax = FMAX[dtype]
    rows, k = x.shape
    xb = x.float().view(rows, k // 32, 32)
    amax = xb.abs().amax(dim=2)
    bits = ((amax / torch.full_like(amax, fmax)).view(torch.int32) + 0x007FFFFF) & 0x7F800000
    inv = torch.where(bits == 0, torch.zeros_like(amax), 1.0 / bits.view(torch.float32))
    q = (xb * inv[:, :, None]).clamp(-fmax, fmax).to(dtype).view(rows, k)
    return q, (bits >> 23).to(torch.uint8)


def _by_chunks(quant, g, rows, k, dtype, std=1.0):
    """Quantised N(0, std) rows, made some rows at a time."""
    step = max(1, (1 << 26) // k)
    parts = [quant(_normal(g, (min(step, rows - r), k), std=std), dtype) for r in range(0, rows, step)]
    return torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts])


def _weights_grouped(g, n, k, dtype, group=128):
    fmax = FMAX[dtype]
    w = _normal(g, (n, k // group, group), std=0.02)
    amax = w.abs().amax(dim=2)
    s = torch.where(amax > 0, amax, torch.ones_like(amax)) / torch.full_like(amax, fmax)
    return (w / s[:, :, None]).clamp(-fmax, fmax).to(dtype).view(n, k), s


def _keys(g, n, nbins, s):
    if s == 0.0:
        return torch.randint(0, nbins, (n,), generator=g, device=DEV, dtype=torch.int32)
    cdf = np.cumsum(np.arange(1, nbins + 1, dtype=np.float64) ** -s)
    cdf = torch.from_numpy(cdf / cdf[-1]).to(DEV)
    u = torch.rand(n, generator=g, device=DEV, dtype=torch.float64)
    return torch.searchsorted(cdf, u, right=True).clamp_(max=nbins - 1).to(torch.int32)


def _offsets(seed, rows, groups):
    w = 1.0 / np.arange(1, groups + 1) ** 0.8
    sizes = np.random.default_rng(int(seed)).multinomial(rows, w / w.sum())
    return torch.from_numpy(np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)).to(DEV)


def prepare(case, seed):
    g = _gen(seed)
    k = case["kind"]
    st = {"case": case}
    if k in ("matmul", "dot_acc"):
        M, N, K, dt = case["M"], case["N"], case["K"], DT[case["dtype"]]
        st["a"] = _normal(g, (M, K), dt)
        st["b"] = _normal(g, (K, N) if case["b"] == "kn" else (N, K), dt)
        if k == "dot_acc":
            st["acc"] = _normal(g, (M, N), std=math.sqrt(K))
    elif k == "fp8_linear":
        st["x"] = _normal(g, (case["M"], case["K"]), torch.bfloat16)
        st["w"], st["sw"] = _by_chunks(_quant_rows, g, case["N"], case["K"], torch.float8_e4m3fn, 0.02)
        st["bias"] = _normal(g, (case["N"],)) if case["bias"] else None
    elif k == "fp8_gemm":
        st["a"], st["sa"] = _by_chunks(_quant_rows, g, case["M"], case["K"], torch.float8_e4m3fn)
        st["b"], st["sb"] = _by_chunks(_quant_rows, g, case["N"], case["K"], torch.float8_e4m3fn)
    elif k == "mx_linear":
        st["x"] = _normal(g, (case["M"], case["K"]), torch.bfloat16)
        st["w"], st["sw"] = _by_chunks(_quant_blocks, g, case["N"], case["K"], DT[case["fmt"]], 0.02)
    elif k == "moe":
        G, N, K = case["G"], case["N"], case["K"]
        st["a"], st["sa"] = _by_chunks(_quant_rows, g, case["rows"], K, torch.float8_e4m3fn)
        w, sw = _by_chunks(_quant_rows, g, G * N, K, torch.float8_e4m3fn, 0.02)
        st["w"], st["sw"] = w.view(G, N, K), sw.view(G, N)
        st["offsets"] = _offsets(seed, case["rows"], G)
    elif k == "gemv":
        st["x"] = _normal(g, (case["M"], case["K"]), torch.bfloat16)
        st["w"], st["sw"] = _weights_grouped(g, case["N"], case["K"], DT[case["fmt"]])
    elif k == "round_trip":
        x = _normal(g, (case["n"],))
        u = torch.empty_like(x).uniform_(-10.0, 5.0, generator=g)
        st["x"] = (x * torch.exp2(u)).to(DT[case["src"]])
    else:
        n = case["n"]
        st["idx"] = _keys(g, n, case["nbins"], case["zipf"])
        st["val"] = (torch.randint(0, 1000, (n,), generator=g, device=DEV, dtype=torch.int32)
                     if case["dtype"] == "int32" else _normal(g, (n,)))
    return st


# ------------------------------------------------------------------ one pass
def run(st):
    case = st["case"]
    k = case["kind"]
    if k == "matmul":
        return tx.matmul(st["a"], st["b"]) if case["b"] == "kn" else tx.dot(st["a"], st["b"])
    if k == "dot_acc":
        return tx.dot_acc(st["a"], st["b"], st["acc"], b_layout=case["b"])
    if k == "fp8_linear":
        q, s = tx.quantize_rowwise(st["x"])
        return tx.dot_scaled_rowcol(q, s, st["w"], st["sw"], bias=st["bias"], activation=case["act"],
                                    out_dtype=DT[case["out"]])
    if k == "fp8_gemm":
        return tx.dot_scaled_rowcol(st["a"], st["sa"], st["b"], st["sb"])
    if k == "mx_linear":
        q, s = tx.quantize_mx(st["x"], DT[case["fmt"]])
        return tx.dot_scaled(q, s, st["w"], st["sw"], out_dtype=DT[case["out"]])
    if k == "moe":
        return tx.dot_scaled_rowcol_grouped(st["a"], st["sa"], st["w"], st["sw"], st["offsets"])
    if k == "gemv":
        return tx.gemv_fp8_dequant(st["x"], st["w"], st["sw"])
    if k == "round_trip":
        q = tx.fp_to_fp(st["x"], DT[case["fmt"]], saturate=case["saturate"])
        return q, tx.fp_to_fp(q, DT[case["src"]])
    bins = torch.zeros(case["nbins"], dtype=DT[case["dtype"]], device=DEV)
    return tx.atomic_rmw("add" if case["dtype"] == "int32" else "fadd", bins, st["idx"], st["val"])


# ------------------------------------------------------------------ what it cannot do without
def work(case):
    k = case["kind"]
    if k in ("matmul", "dot_acc"):
        M, N, K = case["M"], case["N"], case["K"]
        out = 2 * M * N if k == "matmul" else 8 * M * N
        return {"bytes": 2 * (M * K + N * K) + out, "flops": 2 * M * N * K}
    if k in ("fp8_linear", "mx_linear"):
        M, N, K = case["M"], case["N"], case["K"]
        scales = 4 * N if k == "fp8_linear" else N * K // 32
        return {"bytes": 2 * M * K + N * K + scales + (4 * N if case.get("bias") else 0) + SIZE[case["out"]] * M * N,
                "flops": 2 * M * N * K}
    if k == "fp8_gemm":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": (M + N) * (K + 4) + 2 * M * N, "flops": 2 * M * N * K}
    if k == "moe":
        G, M, N, K = case["G"], case["rows"], case["N"], case["K"]
        return {"bytes": M * (K + 4) + min(G, M) * N * (K + 4) + 4 * (G + 1) + 2 * M * N, "flops": 2 * M * N * K}
    if k == "gemv":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": N * K + 4 * N * (K // 128) + 2 * M * K + 2 * M * N, "flops": 2 * M * N * K}
    if k == "round_trip":
        return {"bytes": 2 * (SIZE[case["src"]] + 1) * case["n"], "flops": 2 * case["n"]}
    return {"bytes": 8 * case["n"] + 4 * case["nbins"], "flops": case["n"]}


def tolerance(case):
    k = case["kind"]
    # Codes and integer sums are fixed by the inputs; a scatter's fp32 sums up to their order (6e-7 off
    # the 64-bit sums at most, over 256 .. 1 Mi bins and up to 64 Mi updates).
    if k == "round_trip" or (k == "scatter" and case["dtype"] == "int32"):
        return "exact"
    if k == "scatter":
        return {"rel": 3e-6}
    out = "fp32" if k == "dot_acc" else case.get("out") or ("fp16" if k == "matmul" and case["b"] == "kn" else
                                                            case.get("dtype", "bf16"))
    # About four times the distance to the 64-bit product: the output's rounding (1.7e-3 for bf16, 2.1e-4
    # for fp16), and for fp32 outputs the sums' (1.3e-7 for 16-bit operands, 1.5e-5 inside the fp8 MFMAs,
    # which align a K block's products to its largest).
    return {"rel": {"bf16": 6e-3, "fp16": 8e-4, "fp32": 6e-7 if k == "dot_acc" else 6e-5}[out]}


# ------------------------------------------------------------------ the same in 64 bits
def _act64(y, act):
    if act == "relu":
        return y.clamp(min=0)
    if act == "gelu_tanh":
        return 0.5 * y * (1 + torch.tanh(math.sqrt(2 / math.pi) * (y + 0.044715 * y ** 3)))
    return y / (1 + torch.exp(-y)) if act == "silu" else y


def exact(case, seed):
    st = prepare(case, seed)
    k = case["kind"]
    f64 = torch.float64
    if k in ("matmul", "dot_acc"):
        b = st["b"].to(f64)
        y = st["a"].to(f64) @ (b if case["b"] == "kn" else b.t())
        return y + st["acc"].to(f64) if k == "dot_acc" else y
    if k == "fp8_linear":
        q, s = _quant_rows(st["x"], torch.float8_e4m3fn)
        y = (q.to(f64) @ st["w"].to(f64).t()) * s.to(f64)[:, None] * st["sw"].to(f64)[None, :]
        return _act64(y + st["bias"].to(f64) if case["bias"] else y, case["act"])
    if k == "fp8_gemm":
        return (st["a"].to(f64) @ st["b"].to(f64).t()) * st["sa"].to(f64)[:, None] * st["sb"].to(f64)[None, :]
    if k == "mx_linear":
        q, s = _quant_blocks(st["x"], DT[case["fmt"]])

        def wide(codes, e):
            return codes.to(f64) * torch.exp2(e.to(f64) - 127).repeat_interleave(32, dim=1)
        return wide(q, s) @ wide(st["w"], st["sw"]).t()
    if k == "moe":
        y = torch.empty(case["rows"], case["N"], dtype=f64, device=DEV)
        off = st["offsets"].tolist()
        for p in range(case["G"]):
            lo, hi = off[p], off[p + 1]
            y[lo:hi] = (st["a"][lo:hi].to(f64) @ st["w"][p].to(f64).t()) * st["sw"][p].to(f64)
        return y * st["sa"].to(f64)[:, None]
    if k == "gemv":
        return st["x"].to(f64) @ (st["w"].to(f64) * st["sw"].to(f64).repeat_interleave(128, dim=1)).t()
    if k == "round_trip":
        fmt = DT[case["fmt"]]
        x = st["x"].float()
        q = (x.clamp(-FMAX[fmt], FMAX[fmt]) if case["saturate"] else x).to(fmt)
        return q, q.to(DT[case["src"]])
    bins = np.bincount(st["idx"].cpu().numpy(), weights=st["val"].cpu().numpy(), minlength=case["nbins"])
    if case["dtype"] == "fp32":
        return torch.from_numpy(bins).to(DEV)
    wrapped = (bins.astype(np.int64) + (1 << 31)) % (1 << 32) - (1 << 31)
    return torch.from_numpy(wrapped.astype(np.int32)).to(DEV)
