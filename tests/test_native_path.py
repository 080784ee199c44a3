"""The native call path of ferret_amd.ops (csrc/native.cpp).

It takes the plain case only: on the CPU, everything else must come back as
None, so that the Python path answers it; on the GPU each operator gives the
bits of the Python path, and the errors stay that path's own.
"""
from __future__ import annotations

import os
import shutil
import sys

import pytest
import torch

from ferret_amd import lib


@pytest.fixture(scope="module")
def native():
    if not os.path.exists(lib.LIB_PATH):
        pytest.skip("libferret_hip.so not built")
    return lib.native()


def test_cpu_tensors_and_other_objects_are_not_taken(native):
    x, w = torch.zeros(2, 128, dtype=torch.bfloat16), torch.zeros(16, 128, dtype=torch.bfloat16)
    assert native.linear_bf16(x, w, None, None, None) is None
    assert native.linear_bf16(None, w, None, None, None) is None
    assert native.moe_permute(torch.zeros(2, 2, dtype=torch.int32), "8", None, None) is None
    with pytest.raises(TypeError):
        native.linear_bf16(x, w)


def test_modes_are_left_to_python(native):
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        assert native.quant_act_e4m3(torch.zeros(2, 128, dtype=torch.bfloat16, device="cuda"), None, None) is None


def test_without_the_module_operators_take_the_python_path(native, monkeypatch, tmp_path):
    monkeypatch.setattr(lib, "_NATIVE", None)
    monkeypatch.setattr(lib, "NATIVE_PATH", str(tmp_path / "_native.so"))
    with pytest.warns(RuntimeWarning, match="_native.so is missing"):
        nat = lib.native()
    assert nat.linear_bf16(None, None, None, None, None) is None
    assert lib.native() is nat      # warned of once
    from ferret_amd import ops
    with pytest.raises(ValueError, match="GPU tensor"):
        ops.linear_bf16(torch.zeros(2, 128, dtype=torch.bfloat16), torch.zeros(16, 128, dtype=torch.bfloat16))


@pytest.mark.parametrize("absent", ["torch", "g++"])
def test_the_library_builds_without_what_only_the_module_needs(monkeypatch, tmp_path, absent):
    from ferret_amd import build
    stale = tmp_path / "_native.so"
    stale.write_bytes(b"")
    monkeypatch.setattr(build, "NATIVE", str(stale))
    if absent == "torch":
        monkeypatch.setitem(sys.modules, "torch", None)
    else:
        which = shutil.which
        monkeypatch.setattr(build.shutil, "which", lambda name: None if name == "g++" else which(name))
    assert build.build_native() is None and not stale.exists()


def _moe(ops):
    from ferret_amd import workloads as W
    T, E, H, inter = 37, 6, 256, 256
    g = torch.Generator(device="cuda").manual_seed(3)
    logits = torch.randn((T, E), generator=g, device="cuda")
    x, sx = W.quant_act_1x128(W.randn((T, H), 5, "cuda"))
    ws = []
    for e in range(E):
        ws.append(W.quant_weight_128x128(W.randn((2 * inter, H), 10 + e, "cuda")) +
                  W.quant_weight_128x128(W.randn((H, inter), 30 + e, "cuda")))
    w13, s13, w2, s2 = (torch.stack([w[i].view(torch.uint8) if i % 2 == 0 else w[i] for w in ws]) for i in range(4))
    ids, wt = ops.moe_route_topk(logits, 3)
    rt = ops.moe_permute(ids, E)
    h = ops.moe_w13_fp8(x, sx, w13, s13, rt)
    q, sq = ops.quant_act_e4m3(h)
    o = ops.moe_w2_fp8(q, sq, w2, s2, rt, mma="e4m3")
    wq = torch.randint(-2 ** 31, 2 ** 31, (E, 64, H // 8), generator=g, device="cuda", dtype=torch.int32)
    i4s = (torch.randn((E, 64, H // 32), generator=g, device="cuda") * 0.01).to(torch.bfloat16)
    xb = W.randn((T, H), 6, "cuda").to(torch.bfloat16)
    rt16 = ops.moe_permute(ids, E, 16)
    return [ids, wt, rt.counts, rt.offsets, rt.sorted_pair, rt.tiles, rt.ntiles, h, q, sq, o, ops.moe_combine(o, wt),
            ops.moe_w13_w4a16(xb, wq, i4s, rt16), ops.moe_w13_w4a16(xb, ops.int4_tile_weights(wq), i4s, rt16)]


def _dense(ops):
    from ferret_amd import workloads as W
    out = []
    for M in (3, 40):
        x, w = W.randn((M, 512), 1, "cuda").to(torch.bfloat16), W.randn((256, 512), 2, "cuda").to(torch.bfloat16)
        r, y = W.randn((M, 256), 3, "cuda").to(torch.bfloat16), torch.empty((M, 256), dtype=torch.bfloat16, device="cuda")
        out += [ops.linear_bf16(x, w), ops.linear_bf16(x, w, r, out=y, workspace=torch.empty(8, device="cuda"))]
        a, sa = W.quant_act_1x128(W.randn((M, 512), 4, "cuda"))
        b, sb = W.quant_weight_128x128(W.randn((256, 512), 5, "cuda"))
        out += [ops.fp8_gemm_blockscale(a, sa, b, sb), ops.fp8_gemm_blockscale(a, sa, b, sb, mma="e4m3")]
        sfa = ops.pack_ue8m0(ops.ue8m0_from_float(sa))
        sfb = ops.pack_ue8m0(ops.ue8m0_from_float(ops.expand_block_scales(sb, 256)))
        out.append(ops.fp8_gemm_ue8m0(a, sfa, b, sfb))
    return out


class _Recorder:
    """The native functions, with the names of those that took a call (and those that left one) noted."""

    def __init__(self, nat):
        self.nat, self.took, self.left = nat, set(), set()

    def __getattr__(self, name):
        def call(*args):
            r = getattr(self.nat, name)(*args)
            (self.left if r is None else self.took).add(name)
            return r
        return call


OPERATORS = {
    "_moe": {"moe_route_topk", "moe_permute", "moe_w13_fp8", "quant_act_e4m3", "moe_w2_fp8", "moe_combine",
             "moe_w13_w4a16"},
    "_dense": {"linear_bf16", "fp8_gemm_blockscale", "fp8_gemm_ue8m0"}}


@pytest.mark.gpu
@pytest.mark.parametrize("calls", [_moe, _dense])
def test_gives_the_bits_of_the_python_path(hip, monkeypatch, calls):
    from ferret_amd import ops
    print(f"[case] native path {calls.__name__}", flush=True)
    rec = _Recorder(lib.native())
    monkeypatch.setattr(lib, "native", lambda: rec)
    here = calls(ops)
    assert rec.took == OPERATORS[calls.__name__] and not rec.left
    monkeypatch.setattr(lib, "native", lambda: lib._Absent())
    there = calls(ops)
    torch.cuda.synchronize()
    assert len(here) == len(there)
    for i, (a, b) in enumerate(zip(here, there)):
        assert a.shape == b.shape and a.dtype == b.dtype
        assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8)), i


@pytest.mark.gpu
def test_takes_the_plain_case_and_leaves_the_rest(hip):
    from ferret_amd import ops
    nat = lib.native()
    x, w = (torch.zeros((n, 256), dtype=torch.bfloat16, device="cuda") for n in (4, 32))
    assert nat.linear_bf16(x, w, None, None, None) is not None
    assert nat.linear_bf16(x.float(), w, None, None, None) is None                      # type
    assert nat.linear_bf16(x.t(), w, None, None, None) is None                          # strides
    assert nat.linear_bf16(x, w, None, torch.empty_like(x), None) is None               # shape of out
    assert nat.linear_bf16(x, w, None, None, torch.zeros(4)) is None                    # workspace on the host
    assert nat.linear_bf16(x, w[:, :130].contiguous(), None, None, None) is None        # K
    with pytest.raises(ValueError):
        ops.linear_bf16(x, w, out=torch.empty_like(x))
    with pytest.raises(TypeError):
        ops.linear_bf16(x.float(), w)
    got = []
    torch.func.vmap(lambda v: (got.append(nat.linear_bf16(v, w, None, None, None)), v)[1])(torch.stack([x, x]))
    assert got == [None]
