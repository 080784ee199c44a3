"""The small-tile FP8 product past 16 tokens: edges of its tiles and K splits.

Against the oracle, with a caller's workspace (its splits) and without (unsplit,
here or in the larger tiles), at token counts on both sides of every tile size,
K of one scale block, of an odd number of them and of fewer than the splits.
"""
from __future__ import annotations

import pytest
import torch

from oracle import gemm as G
from tests.gpu_helpers import assert_gemm_close, bf16_out, codes8, f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [
    (17, 128, 128), (32, 4096, 384), (33, 256, 2432), (48, 1152, 128), (64, 7168, 640), (65, 128, 3072), (24, 4096, 7168),
    (96, 384, 1152), (100, 2048, 4224), (128, 4096, 512), (129, 1024, 256), (200, 640, 1664), (256, 256, 3072),
    (31, 7168, 16384), (33, 8320, 128), (33, 1152, 1664), (65, 8320, 256), (65, 1152, 1408),
    # past 256 tokens, never split: every tile, odd block counts, the last shape of one round and the first past it
    (257, 1024, 128), (300, 256, 2432), (1313, 128, 384), (490, 1024, 1152), (512, 2048, 640), (1024, 2048, 512),
    (1025, 2048, 512), (269, 1536, 16384)])
def test_matches_the_oracle(hip, M, N, K):
    from ferret_amd import workloads as W
    print(f"[case] fp8 mid M={M} N={N} K={K}", flush=True)
    a, sa = W.quant_act_1x128(W.randn((M, K), M + K, "cuda"))
    b, sb = W.quant_weight_128x128(W.randn((N, K), N, "cuda"))
    ref = G.fp8_blockscale_gemm(codes8(a), f32(sa), codes8(b), f32(sb))
    need = int(hip.ferret_workspace_bytes(1, M, N, K, 0))
    ws = torch.full((max(need, 1),), 0xFF, dtype=torch.uint8, device="cuda")  # NaN partials if any were not written
    for wp, wn, tag in ((ws.data_ptr(), need, "workspace"), (None, 0, "none")):
        c = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert hip.ferret_fp8_gemm_blockscale(a.data_ptr(), sa.data_ptr(), b.data_ptr(), sb.data_ptr(), c.data_ptr(),
                                              M, N, K, wp, wn, torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        assert_gemm_close(bf16_out(c), ref, f"fp8 mid {tag}")


@pytest.mark.parametrize("M,N,K,splits", [(17, 128, 1408, 4), (100, 512, 1664, 4)])
@pytest.mark.parametrize("mma", ["bf16", "e4m3", "ue8m0"])
def test_workspace_of_the_128_row_tiles(hip, M, N, K, splits, mma):
    """Smaller than the small tiles' partials: the 128 x 128 tiles split K in it, and no byte past it is written."""
    from ferret_amd import lib, ops, workloads as W
    print(f"[case] fp8 small workspace {mma} M={M} N={N} K={K}", flush=True)
    a, sa = W.quant_act_1x128(W.randn((M, K), M + K, "cuda"))
    b, sb = W.quant_weight_128x128(W.randn((N, K), N, "cuda"))
    sfa, sfb = ops.ue8m0_from_float(sa), ops.ue8m0_from_float(ops.expand_block_scales(sb, N))
    size = splits * M * N * 4
    assert size < hip.ferret_workspace_bytes(1, M, N, K, 0)
    if mma == "ue8m0":
        size += int(hip.ferret_workspace_bytes(5, M, N, K, 0)) - int(hip.ferret_workspace_bytes(1, M, N, K, 0))
        sa, sb = (torch.ldexp(torch.ones_like(s, dtype=torch.float32), s.int() - 127) for s in (sfa, sfb[::128].contiguous()))
    ws = torch.full((size + 4096,), 0xFF, dtype=torch.uint8, device="cuda")
    c = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    st = torch.cuda.current_stream().cuda_stream

    def call(n):
        if mma == "ue8m0":
            return hip.ferret_fp8_gemm_ue8m0(a.data_ptr(), words[0].data_ptr(), b.data_ptr(), words[1].data_ptr(),
                                             c.data_ptr(), M, N, K, ws.data_ptr(), n, st)
        return hip.ferret_fp8_gemm_blockscale_ex(a.data_ptr(), sa.data_ptr(), b.data_ptr(), sb.data_ptr(), c.data_ptr(),
                                                 M, N, K, ws.data_ptr(), n, lib.FP8_MMA_E4M3 if mma == "e4m3" else 0, st)

    words = [ops.pack_ue8m0(sfa), ops.pack_ue8m0(sfb)]
    assert call(size) == 0
    torch.cuda.synchronize()
    if mma == "e4m3":  # coarser than the oracle's tolerance: the bits of a call with the whole workspace
        assert torch.equal(c.view(torch.int16), ops.fp8_gemm_blockscale(a, sa, b, sb, mma="e4m3").view(torch.int16))
    else:
        assert_gemm_close(bf16_out(c), G.fp8_blockscale_gemm(codes8(a), f32(sa), codes8(b), f32(sb)), f"fp8 {mma}")
    assert bool((ws[size:] == 0xFF).all())
    assert not bool((ws[size - splits * M * N * 4:size].view(torch.int32) == -1).any())  # every partial was written
    if mma == "ue8m0":
        assert call(size - 4) == -3
