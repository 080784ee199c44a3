"""The LDS-tiled bf16 product: edges of its tiles, its K splits and its entry points.

Against the oracle, at token and row counts on both sides of every tile size,
K that no power of two divides, and K shorter than the splits; then the
allocation-free entry against the workspace one, bit for bit, also where the
partials exceed its array and the product runs in several row ranges.
"""
from __future__ import annotations

import pytest
import torch

from oracle import gemm as G
from oracle import metrics as MT
from tests.gpu_helpers import assert_gemm_close, bf16_out, bits16

pytestmark = pytest.mark.gpu


def _inputs(M, N, K, res):
    g = torch.Generator(device="cuda").manual_seed(M * 1000 + N + K)
    x = torch.randn((M, K), generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn((N, K), generator=g, device="cuda") * 0.05).to(torch.bfloat16)
    return x, w, torch.randn((M, N), generator=g, device="cuda").to(torch.bfloat16) if res else None


# M, N, K, tile, K splits: every tile the plan has, unsplit and split, with remainders of rows and tokens (the rule
# is held to it on the CPU, in test_linear_route.py)
EVERY_TILE = [
    (1, 9200, 1152, 0, 1), (5, 3152, 3328, 0, 5), (1, 16624, 640, 1, 1), (5, 5728, 1920, 1, 4), (17, 10352, 512, 2, 1),
    (17, 3152, 1664, 2, 5), (17, 21056, 256, 3, 1), (17, 2800, 2688, 3, 7), (35, 9200, 384, 4, 1), (35, 480, 7296, 4, 8),
    (35, 16624, 256, 5, 1), (35, 5728, 1536, 5, 4), (50, 10352, 256, 6, 1), (50, 1712, 1536, 6, 6), (50, 21056, 128, 7, 1),
    (50, 2800, 2688, 7, 7), (65, 2800, 768, 8, 1), (65, 912, 2304, 8, 6), (65, 16624, 128, 9, 1), (98, 1184, 1664, 9, 7),
    (98, 14768, 128, 10, 1), (98, 2192, 1408, 10, 6), (1, 30016, 384, 11, 1), (1, 6448, 2176, 11, 5)]

# M: one past a tile, exact, one short, several token tiles.  N: remainders of 16, 48, 64 and 80 in the row tiles.
# K / 128: 1 (fewer steps than stages), 2, 5, 19, 78; up to 16 tokens the shapes the stream kernel leaves.
@pytest.mark.parametrize("M,N,K,res", [
    (17, 49168, 128, True), (32, 12304, 640, False), (33, 2128, 2432, True), (48, 5072, 4096, True),
    (49, 24592, 128, False), (64, 6160, 640, True), (65, 304, 9984, False), (96, 1040, 2432, True),
    (97, 1552, 4096, False), (128, 2064, 640, True), (129, 528, 2432, False), (255, 688, 1280, True),
    (300, 1552, 384, False), (1, 1536, 9984, True), (16, 4400, 2432, False), (7, 25008, 640, True),
    (20, 73744, 256, False), (100, 24592, 256, True), (1001, 208, 2432, False)] +
    [(M, N, K, i % 2 == 0) for i, (M, N, K, _, _) in enumerate(EVERY_TILE)])
def test_matches_the_oracle(ops, M, N, K, res):
    print(f"[case] bf16 tiled M={M} N={N} K={K} res={res}", flush=True)
    x, w, r = _inputs(M, N, K, res)
    y = ops.linear_bf16(x, w, r, out=torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda"))
    torch.cuda.synchronize()
    ref = G.linear_bf16(bits16(x), bits16(w), bits16(r) if res else None)
    assert_gemm_close(bf16_out(y), ref, "bf16 tiled")
    e, nbad = MT.linear_rel_err(bf16_out(y), ref)
    assert nbad == 0 and e < 5e-3


@pytest.mark.parametrize("M,N,K,res", [(20, 4096, 4096, True), (64, 6144, 4096, True), (100, 6144, 4096, False)])
def test_allocation_free_entry_gives_the_same_bits(hip, M, N, K, res):
    need = int(hip.ferret_workspace_bytes(0, M, N, K, 0))
    print(f"[case] bf16 tiled noalloc M={M} N={N} K={K} partials {need}", flush=True)
    assert need > 0 and hip.ferret_linear_bf16_noalloc_max_bytes() == 4 << 20
    x, w, r = _inputs(M, N, K, res)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    ya, yb = (torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    rp, st = r.data_ptr() if res else None, torch.cuda.current_stream().cuda_stream
    assert hip.ferret_linear_bf16(x.data_ptr(), w.data_ptr(), rp, ya.data_ptr(), M, N, K, ws.data_ptr(), need, st) == 0
    assert hip.ferret_linear_bf16_noalloc(x.data_ptr(), w.data_ptr(), rp, yb.data_ptr(), M, N, K, st) == 0
    torch.cuda.synchronize()
    assert torch.equal(ya.view(torch.int16), yb.view(torch.int16))


@pytest.fixture(scope="module")
def ops(hip):
    from ferret_amd import ops as O
    return O


def _at(t, elements):
    """t's values in a contiguous tensor that starts `elements` into its allocation."""
    buf = torch.zeros(t.numel() + elements, dtype=t.dtype, device=t.device)
    v = buf[elements:].view(t.shape)
    v.copy_(t)
    return v


@pytest.mark.parametrize("M,N,K", [(40, 1552, 1280), (64, 6144, 4096), (7, 1536, 9984)])
@pytest.mark.parametrize("which", ["x", "residual", "out"])
def test_unaligned_tensors_keep_the_earlier_kernels(ops, hip, M, N, K, which):
    """Views that start inside a buffer: x 8 bytes past a 16-byte bound, residual or y 2 bytes past one."""
    print(f"[case] bf16 linear unaligned {which} M={M} N={N} K={K}", flush=True)
    x, w, r = _inputs(M, N, K, True)
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    ref = G.linear_bf16(bits16(x), bits16(w), bits16(r))
    x, r, y = (_at(t, 0 if which != name else 4 if name == "x" else 1)
               for t, name in ((x, "x"), (r, "residual"), (y, "out")))
    ops.linear_bf16(x, w, r, out=y)
    torch.cuda.synchronize()
    assert_gemm_close(bf16_out(y), ref, f"unaligned {which}")
    y.fill_(float("nan"))
    assert hip.ferret_linear_bf16_noalloc(x.data_ptr(), w.data_ptr(), r.data_ptr(), y.data_ptr(), M, N, K,
                                          torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert_gemm_close(bf16_out(y), ref, f"unaligned {which}, allocation-free entry")


@pytest.mark.parametrize("M,N,K,splits", [(48, 4096, 12288, 3), (64, 1536, 12288, 6)])
def test_workspace_of_the_16_token_split(hip, M, N, K, splits):
    """Smaller than the tiled plan's partials: the 16-token kernels split K in it, and write no byte past it."""
    size = splits * M * N * 4
    print(f"[case] bf16 linear small workspace M={M} N={N} K={K} bytes {size}", flush=True)
    assert size < hip.ferret_workspace_bytes(0, M, N, K, 0)
    x, w, r = _inputs(M, N, K, True)
    ws = torch.full((size + 4096,), 0xFF, dtype=torch.uint8, device="cuda")
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    assert hip.ferret_linear_bf16(x.data_ptr(), w.data_ptr(), r.data_ptr(), y.data_ptr(), M, N, K, ws.data_ptr(), size,
                                  torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert_gemm_close(bf16_out(y), G.linear_bf16(bits16(x), bits16(w), bits16(r)), "small workspace")
    assert bool((ws[size:] == 0xFF).all())
    assert not bool((ws[:size].view(torch.int32) == -1).any())   # every partial was written


def _workspace_bits(hip, x, w, r, M, N, K):
    need = int(hip.ferret_workspace_bytes(0, M, N, K, 0))
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device="cuda")
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    assert need > 0 and hip.ferret_linear_bf16(
        x.data_ptr(), w.data_ptr(), r.data_ptr() if r is not None else None, y.data_ptr(), M, N, K, ws.data_ptr(),
        need, torch.cuda.current_stream().cuda_stream) == 0
    return y


# One shape per tile and token-tile count that splits K where the 16-token kernels did not (these run without the
# library's array), then shapes whose 16-token split uses it: partials that fit, and row ranges.
@pytest.mark.parametrize("M,N,K,res", [
    (5, 4096, 2560, True), (5, 4320, 2432, False), (20, 1008, 5248, True), (20, 4272, 1280, False),
    (33, 1440, 2432, True), (33, 3280, 1664, False), (50, 1584, 1664, True), (50, 4224, 1280, False),
    (70, 1824, 1152, True), (100, 592, 2560, False), (70, 3360, 1280, True), (100, 1648, 1280, False),
    (100, 2144, 1408, True), (97, 2720, 1152, True), (200, 1008, 2816, False), (5, 6448, 2176, True),
    (200, 2704, 1792, False), (6, 7616, 1664, True), (2, 10304, 3072, False), (25, 6368, 7168, True), (4, 6352, 2560, True),
    (48, 4096, 12288, True), (64, 4096, 12288, True), (80, 4096, 12288, False)])
def test_allocation_free_entry_gives_the_same_bits_on_every_tile(hip, M, N, K, res):
    print(f"[case] bf16 tiled noalloc M={M} N={N} K={K} res={res}", flush=True)
    x, w, r = _inputs(M, N, K, res)
    want = _workspace_bits(hip, x, w, r, M, N, K)
    hip.ferret_linear_bf16_noalloc_max_bytes()
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    assert hip.ferret_linear_bf16_noalloc(x.data_ptr(), w.data_ptr(), r.data_ptr() if res else None, y.data_ptr(),
                                          M, N, K, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))


def test_allocation_free_calls_without_a_16_token_split_may_overlap(hip):
    """Two streams at once, shapes whose 16-token split is one: no memory is shared."""
    shapes = [(64, 4096, 4096), (8, 1536, 9984)]
    print("[case] bf16 tiled noalloc on two streams", flush=True)
    ins = [_inputs(*s, False) for s in shapes]
    want = [_workspace_bits(hip, x, w, None, *s) for s, (x, w, _) in zip(shapes, ins)]
    outs = [[torch.empty((M, N), dtype=torch.bfloat16, device="cuda") for _ in range(20)] for M, N, _ in shapes]
    streams = [torch.cuda.Stream() for _ in shapes]
    torch.cuda.synchronize()
    for i in range(20):
        for (M, N, K), (x, w, _), out, st in zip(shapes, ins, outs, streams):
            assert hip.ferret_linear_bf16_noalloc(x.data_ptr(), w.data_ptr(), None, out[i].data_ptr(), M, N, K,
                                                  st.cuda_stream) == 0
    torch.cuda.synchronize()
    for out, y in zip(outs, want):
        assert all(torch.equal(o.view(torch.int16), y.view(torch.int16)) for o in out)


@pytest.mark.parametrize("M,N,K,off", [(512, 4096, 6144, 4), (64, 8192, 6144, 4), (64, 8192, 6144, 0)])
def test_default_workspace_serves_both_kernels(ops, hip, M, N, K, off):
    """Shapes that the tiled plan splits less than the 16-token kernels, through the entry point that allocates."""
    on, any_ = (int(hip.ferret_workspace_bytes(op, M, N, K, 0)) for op in (6, 0))
    print(f"[case] bf16 default workspace M={M} N={N} K={K} off={off} bytes {on} {any_}", flush=True)
    assert on < any_ == 3 * M * N * 4
    x, w, r = _inputs(M, N, K, True)
    y = ops.linear_bf16(_at(x, off), w, r)
    torch.cuda.synchronize()
    assert_gemm_close(bf16_out(y), G.linear_bf16(bits16(x), bits16(w), bits16(r)), "default workspace")
