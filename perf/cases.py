"""The calls that a program built on ferret_amd makes, as cases to time and compare.

Five kinds, each through the public entry points of ferret_amd.ops:

  linear   y = x.W^T (+ residual), bf16: the projections of a decode step.
  fp8      block-scaled e4m3 GEMM, from one decode token to a prefill chunk.
  ue8m0    the same with packed power-of-two scales.
  moe      a whole FP8 MoE layer: top-k routing, permutation, w13 + SiLU, the
           1x128 quantizer, w2 and the weighted combine.
  int4     the W4A16 MoE gate-up projection with its routing and permutation.

Sizes are those of ferret_amd.workloads (Qwen3-8B decode projections,
DeepSeek-V3 dense, attention and MoE shapes, Kimi-K2 INT4), with batch sizes a
server meets between them, ragged ones among them.  Outputs and workspaces are
left to the entry points' defaults (torch's caching allocator).
"""
import math

import torch

from ferret_amd import ops

FP8 = torch.float8_e4m3fn
DEV = "cuda"


def listed():
    return [
        # One token of one sequence through the QKV projection: latency and launches.
        {"name": "linear_qkv_M1", "kind": "linear", "M": 1, "N": 6144, "K": 4096, "residual": False},
        # The down projection of a decode batch of 48 sequences, its residual added.
        {"name": "linear_down_M48_res", "kind": "linear", "M": 48, "N": 4096, "K": 12288, "residual": True},
        # A small decode batch through one rank's FP8 attention output projection.
        {"name": "fp8_oproj_M8", "kind": "fp8", "M": 8, "N": 7168, "K": 2048, "mma": "bf16"},
        # A ragged decode batch through the dense FP8 projection.
        {"name": "fp8_dense_M100", "kind": "fp8", "M": 100, "N": 4096, "K": 7168, "mma": "bf16"},
        # A prefill chunk of a ragged prompt through one rank's q_b projection.
        {"name": "fp8_qb_M1000", "kind": "fp8", "M": 1000, "N": 3072, "K": 1536, "mma": "bf16"},
        # A full prefill batch through the dense FP8 projection.
        {"name": "fp8_dense_M4096", "kind": "fp8", "M": 4096, "N": 4096, "K": 7168, "mma": "bf16"},
        # A ragged prefill batch with power-of-two block scales.
        {"name": "ue8m0_oproj_M3000", "kind": "ue8m0", "M": 3000, "N": 7168, "K": 2048},
        # One MoE layer of a decode step of 128 sequences: every expert's weights are read.
        {"name": "moe_decode_T128", "kind": "moe", "T": 128, "E": 256, "topk": 8, "hidden": 7168, "inter": 2048,
         "zipf": 0.0},
        # The same layer for a large decode batch or a short prefill chunk: a few dozen rows per expert.
        {"name": "moe_chunk_T700", "kind": "moe", "T": 700, "E": 256, "topk": 8, "hidden": 7168, "inter": 2048,
         "zipf": 0.0},
        # The same layer for a prefill batch whose experts are used unevenly.
        {"name": "moe_prefill_T4096", "kind": "moe", "T": 4096, "E": 256, "topk": 8, "hidden": 7168, "inter": 2048,
         "zipf": 1.1},
        # The INT4 gate-up projection of a decode step of 64 sequences, weights tiled at load time.
        {"name": "int4_decode_T64", "kind": "int4", "T": 64, "E": 384, "topk": 8, "N": 4096, "K": 7168, "tiled": True},
        # One tensor-parallel rank of it for a 512-token prompt chunk.
        {"name": "int4_rank_T512", "kind": "int4", "T": 512, "E": 384, "topk": 8, "N": 512, "K": 7168, "tiled": True},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "fp8", "fp8", "fp8", "ue8m0", "moe", "moe", "int4"])
    if kind == "linear":
        M = _log_int(rng, 1, 128)
        if rng.random() < 0.6:
            N, K = rng.choice([(6144, 4096), (4096, 4096), (24576, 4096), (4096, 12288)])
        else:
            N, K = 16 * _log_int(rng, 64, 1536), 128 * _log_int(rng, 8, 96)
        return {"kind": kind, "M": M, "N": N, "K": K, "residual": rng.random() < 0.4}
    if kind in ("fp8", "ue8m0"):
        M = _log_int(rng, 1 if kind == "fp8" else 32, 8192)
        if rng.random() < 0.6:
            N, K = rng.choice([(4096, 7168), (3072, 1536), (4096, 512), (7168, 2048)])
        else:
            N, K = 128 * _log_int(rng, 8, 56), 128 * _log_int(rng, 4, 56)
        case = {"kind": kind, "M": M, "N": N, "K": K}
        if kind == "fp8":
            case["mma"] = "e4m3" if rng.random() < 0.15 else "bf16"
        return case
    if kind == "moe":
        E = rng.choice([32, 64, 256])
        return {"kind": kind, "T": _log_int(rng, 1, 4096), "E": E, "topk": rng.choice([1, 2, 4, 8, 8, 8]),
                "hidden": rng.choice([2048, 4096, 7168]), "inter": rng.choice([768, 1536, 2048]),
                "zipf": rng.choice([0.0, 0.0, 1.1])}
    return {"kind": kind, "T": _log_int(rng, 1, 1024), "E": 384, "topk": 8, "N": rng.choice([512, 1024, 4096]),
            "K": rng.choice([4096, 7168]), "tiled": rng.random() < 0.75}


# ------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV)


def _quant_rows(x):
    """1x128 absmax / 448 blocks of activations."""
    M, K = x.shape
    v = x.view(M, K // 128, 128)
    amax = v.abs().amax(2).clamp_min(1e-4)
    return (v * (448.0 / amax).unsqueeze(2)).to(FP8).view(M, K), amax / 448.0


def _quant_blocks(w):
    """128x128 absmax / 448 blocks of weights [..., N, K]."""
    *b, N, K = w.shape
    v = w.view(*b, N // 128, 128, K // 128, 128)
    amax = v.abs().amax((-3, -1)).clamp_min(1e-6)
    q = v.mul_((448.0 / amax).unsqueeze(-2).unsqueeze(-1)).to(FP8).view(*b, N, K)
    return q, amax / 448.0


def _pow2_quant(x, scale, spread):
    """e4m3 codes of x under its block scales rounded to powers of two, and those scales' UE8M0 bytes."""
    ue = ops.ue8m0_from_float(scale)
    step = torch.exp2(ue.float() - 127.0)
    return (x / spread(step)).clamp(-448.0, 448.0).to(FP8), ue


def _moe_weights(g, E, N, K):
    w = torch.empty((E, N, K), dtype=FP8, device=DEV)
    sw = torch.empty((E, N // 128, K // 128), device=DEV)
    for e in range(0, E, 16):
        w[e:e + 16], sw[e:e + 16] = _quant_blocks(_randn(g, min(16, E - e), N, K))
    return w, sw


def _int4_weights(g, E, N, K):
    """Group-32 absmax / 7 quantized Gaussian weights: packed words (low nibble first) and bf16 scales."""
    wq = torch.empty((E, N, K // 8), dtype=torch.int32, device=DEV)
    ws = torch.empty((E, N, K // 32), dtype=torch.bfloat16, device=DEV)
    shift = (4 * torch.arange(8, device=DEV, dtype=torch.int32))
    for e in range(0, E, 16):
        n = min(16, E - e)
        w = _randn(g, n, N, K // 32, 32).mul_(0.02)
        s = (w.abs().amax(3) / 7.0).to(torch.bfloat16)
        ws[e:e + n] = s
        q = w.div_(s.float().unsqueeze(3)).round_().clamp_(-8, 7).add_(8).to(torch.int32)
        q = (q.view(n, N, K // 8, 8) << shift)
        wq[e:e + n] = q.sum(3, dtype=torch.int32)  # disjoint bits: the sum is the packed word
    return wq, ws


def _logits(g, T, E, zipf):
    if not zipf:
        return _randn(g, T, E)
    u = torch.rand((T, E), generator=g, device=DEV).clamp(1e-12, 1.0 - 1e-7)
    rank = torch.arange(1, E + 1, device=DEV, dtype=torch.float32)
    return -torch.log(-torch.log(u)) - zipf * torch.log(rank)


def prepare(case, seed):
    g = _gen(seed)
    s = {"case": case}
    kind = case["kind"]
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        s["x"] = _randn(g, M, K).to(torch.bfloat16)
        s["w"] = (_randn(g, N, K) * 0.02).to(torch.bfloat16)
        s["r"] = _randn(g, M, N).to(torch.bfloat16) if case["residual"] else None
    elif kind == "fp8":
        s["a"], s["sa"] = _quant_rows(_randn(g, case["M"], case["K"]))
        s["b"], s["sb"] = _quant_blocks(_randn(g, case["N"], case["K"]))
    elif kind == "ue8m0":
        M, N, K = case["M"], case["N"], case["K"]
        x, w = _randn(g, M, K), _randn(g, N, K)
        sx = x.view(M, K // 128, 128).abs().amax(2) / 448.0
        sw = w.view(N // 128, 128, K // 128, 128).abs().amax((1, 3)) / 448.0
        s["a"], ua = _pow2_quant(x, sx, lambda t: t.repeat_interleave(128, 1))
        s["b"], ub = _pow2_quant(w, sw, lambda t: t.repeat_interleave(128, 1).repeat_interleave(128, 0))
        s["sfa"], s["sfb"] = ops.pack_ue8m0(ua), ops.pack_ue8m0(ops.expand_block_scales(ub, N))
    elif kind == "moe":
        T, E, H, inter = case["T"], case["E"], case["hidden"], case["inter"]
        s["logits"] = _logits(g, T, E, case["zipf"])
        s["x"], s["sx"] = _quant_rows(_randn(g, T, H))
        s["w13"], s["s13"] = _moe_weights(g, E, 2 * inter, H)
        s["s13"] *= 0.02  # gate and up of order one, as trained weights give them
        s["w2"], s["s2"] = _moe_weights(g, E, H, inter)
        s["s2"] *= 0.02
    else:
        T, E, N, K = case["T"], case["E"], case["N"], case["K"]
        s["logits"] = _randn(g, T, E)
        s["x"] = _randn(g, T, K).to(torch.bfloat16)
        wq, s["ws"] = _int4_weights(g, E, N, K)
        s["w"] = ops.int4_tile_weights(wq) if case["tiled"] else wq
    return s


# ------------------------------------------------------------------ the calls

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "linear":
        return ops.linear_bf16(s["x"], s["w"], s["r"])
    if kind == "fp8":
        return ops.fp8_gemm_blockscale(s["a"], s["sa"], s["b"], s["sb"], mma=case["mma"])
    if kind == "ue8m0":
        return ops.fp8_gemm_ue8m0(s["a"], s["sfa"], s["b"], s["sfb"])
    ids, weights = ops.moe_route_topk(s["logits"], case["topk"])
    if kind == "int4":
        rt = ops.moe_permute(ids, case["E"], 16)  # the W4A16 kernels take 16-row tiles
        return {"ids": ids, "weights": weights, "h": ops.moe_w13_w4a16(s["x"], s["w"], s["ws"], rt)}
    rt = ops.moe_permute(ids, case["E"])
    h = ops.moe_w13_fp8(s["x"], s["sx"], s["w13"], s["s13"], rt)
    q, sq = ops.quant_act_e4m3(h)
    o = ops.moe_w2_fp8(q, sq, s["w2"], s["s2"], rt)
    return {"ids": ids, "weights": weights, "h": h, "o": o, "y": ops.moe_combine(o, weights)}


# ------------------------------------------------------------------ what a pass cannot do without

def _hit(case):
    """Experts that a routing of the case is expected to use."""
    E, k, T = case["E"], case["topk"], case["T"]
    p = [(e + 1.0) ** -case.get("zipf", 0.0) for e in range(E)]
    total = sum(p)
    return sum(1.0 - (1.0 - min(1.0, k * x / total)) ** T for x in p)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 2 * (N * K + M * K + M * N * (2 if case["residual"] else 1)), "flops": 2 * M * N * K}
    if kind in ("fp8", "ue8m0"):
        M, N, K = case["M"], case["N"], case["K"]
        nk = K // 128
        scales = 4 * nk * (M + (N + 127) // 128) if kind == "fp8" else 4 * ((nk + 3) // 4) * (M + N)
        return {"bytes": M * K + N * K + scales + 2 * M * N, "flops": 2 * M * N * K}
    T, E, P = case["T"], case["E"], case["T"] * case["topk"]
    route = 4 * T * E + 8 * P
    if kind == "int4":
        N, K = case["N"], case["K"]
        return {"bytes": route + _hit(case) * (N * K // 2 + 2 * N * (K // 32)) + 2 * T * K + P * N,
                "flops": 2 * P * N * K}
    H, inter = case["hidden"], case["inter"]
    return {"bytes": route + _hit(case) * 3 * inter * H + T * H + 2 * P * inter + 2 * P * H + 2 * T * H,
            "flops": 2 * P * 3 * inter * H}


# ------------------------------------------------------------------ tolerance and the 64-bit values

def tolerance(case):
    # Products of bf16 / e4m3 values are exact in fp32 and the outputs are rounded to bf16 once: another order
    # of the fp32 sums moves 0.01-0.05 % of the outputs across a rounding boundary, by one unit in the last
    # place (2^-7 of the value at most).  Measured against the 64-bit values rounded to bf16: rel <= 4.0e-5,
    # max <= 7.8e-3 over the listed and drawn GEMMs.
    if case["kind"] == "moe":
        # A moved h takes its neighbouring e4m3 code (up to 1/8 of its value) into every output of its row:
        # rel 2.3e-3 - 3.1e-3, max 0.03 - 0.11 on o and y.
        return {"rel": 1e-2, "max": 0.4}
    if case.get("mma") == "e4m3":
        return {"rel": 9e-4, "max": 2e-2}  # the FP8 MFMA drops low bits of each group of products: rel 2.3e-4
    return {"rel": 1.6e-4, "max": 2e-2}


def _wide(q, s):
    """Block-scaled codes [R, K] as float64; s: one scale per 128 columns and per row or 128 rows."""
    R, K = q.shape
    s = s.double().repeat_interleave(128, 1)
    if s.shape[0] != R:
        s = s.repeat_interleave(128, 0)[:R]
    return q.to(torch.float32).double() * s


def _bytes(words, nk):
    """Packed UE8M0 words [ceil(nk/4), D] -> scales [D, nk]."""
    b = torch.stack([(words >> (8 * j)) & 0xFF for j in range(4)], 2)  # [nsk, D, 4]
    b = b.permute(1, 0, 2).reshape(words.shape[1], -1)[:, :nk].double()
    return torch.where(b > 0, torch.exp2(b - 127.0), torch.zeros_like(b))


def _route(logits, topk):
    order = torch.sort(logits, dim=1, descending=True, stable=True)[1][:, :topk]
    return order, torch.softmax(logits.double(), 1).gather(1, order)


def _silu(v):
    half = v.shape[1] // 2
    return v[:, :half] * torch.sigmoid(v[:, :half]) * v[:, half:]


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "linear":
        y = s["x"].double() @ s["w"].double().t()
        return y if s["r"] is None else y + s["r"].double()
    if kind == "fp8":
        return _wide(s["a"], s["sa"]) @ _wide(s["b"], s["sb"]).t()
    if kind == "ue8m0":
        nk = case["K"] // 128
        return _wide(s["a"], _bytes(s["sfa"], nk)) @ _wide(s["b"], _bytes(s["sfb"], nk)).t()
    T, E, k = case["T"], case["E"], case["topk"]
    ids, weights = _route(s["logits"], k)
    pair_expert = ids.reshape(-1)
    pairs = [torch.nonzero(pair_expert == e).flatten() for e in range(E)]
    if kind == "int4":
        N, K = case["N"], case["K"]
        h = torch.empty((T * k, N // 2), dtype=torch.float64, device=DEV)
        shift = 4 * torch.arange(8, device=DEV, dtype=torch.int32)
        for e, p in enumerate(pairs):
            if p.numel():
                w = s["w"][e]
                if case["tiled"]:
                    w = w.permute(0, 2, 1, 3).reshape(N, K // 8)
                q = ((w.unsqueeze(2) >> shift) & 15).view(N, K).float() - 8.0
                w = (q * s["ws"][e].float().repeat_interleave(32, 1)).to(torch.bfloat16)  # the format's bf16 weights
                h[p] = _silu(s["x"][p // k].double() @ w.double().t())
        return {"ids": None, "weights": weights, "h": h}
    H, inter = case["hidden"], case["inter"]
    x = _wide(s["x"], s["sx"])
    h = torch.empty((T * k, inter), dtype=torch.float64, device=DEV)
    for e, p in enumerate(pairs):
        if p.numel():
            h[p] = _silu(x[p // k] @ _wide(s["w13"][e], s["s13"][e]).t())
    q, sq = _quant_rows(h.to(torch.bfloat16).float())  # h is handed on in bf16
    o = torch.empty((T * k, H), dtype=torch.float64, device=DEV)
    for e, p in enumerate(pairs):
        if p.numel():
            o[p] = _wide(q[p], sq[p]) @ _wide(s["w2"][e], s["s2"][e]).t()
    y = (o.to(torch.bfloat16).double().view(T, k, H) * weights.unsqueeze(2)).sum(1)
    return {"ids": None, "weights": weights, "h": h, "o": o, "y": y}
