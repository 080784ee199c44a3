"""The INT4 w13 kernel that takes two 16-row tiles of an expert at a time.

The same routed rows go through it and, with the expert count padded by empty
experts until the average falls below its rule, through the one-tile kernels.
Both add an output's products in the same order, so the results must agree bit
for bit, on either weight layout; the small cases are also held to the oracle.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import gemm as G
from tests.gpu_helpers import assert_gemm_close, bf16_out, bits16
from tests.test_linear_route import run_rules

pytestmark = pytest.mark.gpu

EDGES = [1, 15, 16, 17, 0, 31, 32, 33, 48, 49, 64]  # one tile, exactly two, one row into the third


def _rows(E):
    """Edge counts first, then experts of 1 .. 40 rows (more than one round of the table walk for E = 600)."""
    return EDGES + [int(n) for n in np.random.default_rng(E).integers(1, 41, E - len(EDGES))]


@pytest.fixture(scope="module")
def ops(hip):
    from ferret_amd import ops as O
    return O


@pytest.mark.parametrize("E,N,K", [(128, 1024, 128), (128, 1024, 256), (64, 2048, 384),  # as few stages as the ring
                                   (600, 256, 2048), (130, 1024, 2048),                  # a long table; the stream kernel's K
                                   (64, 2048, 2432),                                     # ragged last span
                                   (33, 4096, 7168),
                                   (8, 1024, 2048), (8, 2560, 7168)])                    # few experts of many rows
def test_two_tiles_equal_one(ops, tmp_path, E, N, K):
    rows = _rows(E) if E > 8 else [n * 24 for n in EDGES[:8]]
    P = sum(rows)
    streams = K in (2048, 7168)  # the K of the stream kernel: 14 (tiled) or 16 rows per expert, else 4
    padded = P // (14 if streams else 4) + 1
    print(f"[case] int4 two tiles E={E} P={P} N={N} K={K}", flush=True)
    assert padded <= 1024
    # tiled weights, then the checkpoint layout, whose line lies higher for the stream kernel's larger K
    for is_tiled, taken in ((1, 1), (0, (E, K) != (33, 7168))):
        run_rules(tmp_path, f"CHECK(i4::takes({P}, {E}, {N}, {K // 128}, 4096, 256, {int(streams)}, {is_tiled}) == {int(taken)});"
                            f"CHECK(!i4::takes({P}, {padded}, {N}, {K // 128}, 4096, 256, {int(streams)}, {is_tiled}));",
                  "int4_moe.hpp")
    ids = np.concatenate([np.full(n, e, dtype=np.int32) for e, n in enumerate(rows)])
    np.random.default_rng(E).shuffle(ids)
    ids = torch.from_numpy(ids.reshape(-1, 1)).cuda()
    g = torch.Generator(device="cuda").manual_seed(E + N + K)
    x = torch.randn((P, K), generator=g, device="cuda").to(torch.bfloat16)
    wq = torch.zeros((padded, N, K // 8), dtype=torch.int32, device="cuda")
    wq[:E] = torch.randint(-2 ** 31, 2 ** 31, (E, N, K // 8), generator=g, device="cuda", dtype=torch.int32)
    ws = torch.zeros((padded, N, K // 32), dtype=torch.bfloat16, device="cuda")
    ws[:E] = (torch.randn((E, N, K // 32), generator=g, device="cuda") * 0.01).to(torch.bfloat16)
    rt, rt_padded = ops.moe_permute(ids, E, 16), ops.moe_permute(ids, padded, 16)
    tiled = ops.int4_tile_weights(wq)
    got = None
    for w in (wq, tiled):
        one = ops.moe_w13_w4a16(x, w, ws, rt_padded)
        got = ops.moe_w13_w4a16(x, w[:E], ws[:E], rt,
                                out=torch.full((P, N // 2), float("nan"), dtype=torch.bfloat16, device="cuda"))
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int16), one.view(torch.int16))
    if K <= 256:
        ref = G.moe_w13_w4a16(bits16(x), wq[:E].cpu().numpy(), bits16(ws[:E]), ids.cpu().numpy())
        assert_gemm_close(bf16_out(got), ref, f"N={N} K={K}")


def test_misaligned_scales_keep_the_one_tile_kernel(ops):
    E, N, K, T = 64, 2048, 384, 128  # scales 2 bytes past a word: at any number of rows per expert
    print("[case] int4 two tiles, misaligned scales", flush=True)
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn((T, K), generator=g, device="cuda").to(torch.bfloat16)
    wq = torch.randint(-2 ** 31, 2 ** 31, (E, N, K // 8), generator=g, device="cuda", dtype=torch.int32)
    buf = (torch.randn((E * N * K // 32 + 1,), generator=g, device="cuda") * 0.01).to(torch.bfloat16)
    ws = buf[1:].view(E, N, K // 32)
    ids, _ = ops.moe_route_topk(torch.randn((T, E), generator=g, device="cuda"), 8)
    rt = ops.moe_permute(ids, E, 16)
    assert torch.equal(ops.moe_w13_w4a16(x, wq, ws, rt).view(torch.int16),
                       ops.moe_w13_w4a16(x, wq, ws.clone(), rt).view(torch.int16))
