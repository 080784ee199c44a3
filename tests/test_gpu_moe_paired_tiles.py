"""The FP8 MoE stream kernel that takes two 16-row tiles of an expert per unit.

The same routed rows go through the paired kernel and, with the expert count
padded by empty experts until the average falls below its rule, through the
one-tile kernel.  Both add an output's products in the same order, so the
results must agree bit for bit; the paired one is also held to the oracle.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import gemm as G
from tests.gpu_helpers import assert_gemm_close, bf16_out, codes8, f32
from tests.test_linear_route import run_rules

pytestmark = pytest.mark.gpu

# one tile, exactly two, one row into the third, an odd and an even tile count; then a table past 512 rows
# (two rounds of the table walk) whose runs cross its 64-row chunks
EDGES = [1, 15, 16, 17, 0, 31, 32, 33, 48, 49, 64]
MANY = [int(n) for n in np.random.default_rng(1).integers(1, 31, 600)]


@pytest.fixture(scope="module")
def ops(hip):
    from ferret_amd import ops as O
    return O


def _ids(rows):
    ids = np.concatenate([np.full(n, e, dtype=np.int32) for e, n in enumerate(rows)])
    np.random.default_rng(len(rows)).shuffle(ids)
    return torch.from_numpy(ids.reshape(-1, 1)).cuda()


def _weights(E, N, K, padded):
    from ferret_amd import workloads as W
    w = torch.zeros((padded, N, K), dtype=torch.float8_e4m3fn, device="cuda")
    sw = torch.ones((padded, N // 128, K // 128), dtype=torch.float32, device="cuda")
    for e in range(E):
        w[e], sw[e] = W.quant_weight_128x128(W.randn((N, K), 40 + e, "cuda"))
    return w, sw


# the sizes fill the CUs twice to sixteen times with units, as the rule of the paired kernel asks
@pytest.mark.parametrize("which,rows,N,K", [
    ("w13", EDGES, 6144, 2048), ("w13", EDGES, 3072, 4096), ("w13", EDGES, 3072, 7168), ("w13", MANY, 256, 2048),
    ("w2", EDGES, 12032, 1024), ("w2", EDGES, 3072, 2048), ("w2", EDGES, 3200, 3584), ("w2", MANY, 512, 1024),
    # K / 128 of 12 (3 K-steps per wave), then 4, 6 and 14 (two work-groups of 2 waves per CU)
    ("w2", EDGES, 3072, 1536), ("w2", EDGES, 12032, 512), ("w2", EDGES, 3072, 768), ("w2", EDGES, 3200, 1792),
    ("w2", MANY, 128, 768)])
def test_two_tiles_per_unit_equal_one(ops, tmp_path, which, rows, N, K):
    from ferret_amd import workloads as W
    E, P = len(rows), sum(rows)
    padded = min(1024, P // 6 + 1)
    print(f"[case] paired tiles {which} E={E} P={P} N={N} K={K}", flush=True)
    run_rules(tmp_path, f"CHECK(moe::{which}_pairs({P}, {E}, {N}, {K // 128}, 256));"
                        f"CHECK(!moe::{which}_pairs({P}, {padded}, {N}, {K // 128}, 256));", "moe_plan.hpp")
    ids = _ids(rows)
    x, sx = W.quant_act_1x128(W.randn((P, K), 11, "cuda"))
    w, sw = _weights(E, N, K, padded)
    fn = ops.moe_w13_fp8 if which == "w13" else ops.moe_w2_fp8
    got = fn(x, sx, w[:E], sw[:E], ops.moe_permute(ids, E, 16),
             out=torch.full((P, N // 2 if which == "w13" else N), float("nan"), dtype=torch.bfloat16, device="cuda"))
    one = fn(x, sx, w, sw, ops.moe_permute(ids, padded, 16))
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), one.view(torch.int16))
    if E < 100:
        oracle = G.moe_w13_fp8 if which == "w13" else G.moe_w2_fp8
        ref = oracle(codes8(x), f32(sx), codes8(w[:E]), f32(sw[:E]), ids.cpu().numpy())
        assert_gemm_close(bf16_out(got), ref, f"{which} N={N} K={K}")


@pytest.mark.parametrize("N,K", [(2048, 1536), (16384, 512), (6144, 768), (6144, 1792)])
def test_w2_weights_off_a_16_byte_bound(ops, tmp_path, N, K):
    """K / 128 = 12, 4, 6 and 14: weights that start 8 bytes into a buffer keep the per-unit kernel."""
    from ferret_amd import workloads as W
    E, P = 6, 40
    units = ops.moe_permute(torch.zeros((P, 1), dtype=torch.int32, device="cuda"), E, 16).max_tiles * (N // 64)
    run_rules(tmp_path, f"CHECK(moe::w2_streams({K // 128}, (void*)64, {units}, 256));", "moe_plan.hpp")
    print(f"[case] w2 unaligned weights K={K}", flush=True)
    ids = torch.arange(P, device="cuda", dtype=torch.int32).remainder(E).view(-1, 1).contiguous()
    x, sx = W.quant_act_1x128(W.randn((P, K), 11, "cuda"))
    w, sw = _weights(E, N, K, E)
    buf = torch.zeros(w.numel() + 8, dtype=torch.uint8, device="cuda")
    off = buf[8:].view(w.shape)
    off.copy_(w.view(torch.uint8))
    got = ops.moe_w2_fp8(x, sx, off, sw, ops.moe_permute(ids, E, 16))
    torch.cuda.synchronize()
    ref = G.moe_w2_fp8(codes8(x), f32(sx), codes8(w), f32(sw), ids.cpu().numpy())
    assert_gemm_close(bf16_out(got), ref, f"w2 unaligned K={K}")
