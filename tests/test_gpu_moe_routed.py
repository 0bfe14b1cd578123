"""Expert layers of few slots: the decode kernel finds its rows in topk_ids itself (sonar_moe_routed_gemm) and forms the gated activation
where its rows end.  Every form against the layer with sorted slots and an activation of its own, whose bits it has, but where
gate and up halves share a workgroup and K is dealt to half as many wavefronts; and routings that no sorting prepared: experts out of
range, an expert twice for a token, all slots on one, each number of slots around the ballots' 64."""
from __future__ import annotations

import ctypes
import hashlib
import os
import subprocess
import sys

import pytest
import torch

from sonar_amd import _lib, fused_moe
from sonar_amd.scalar_type import scalar_types

DEV = "cuda:0"
BITS = {torch.float16: 11, torch.bfloat16: 8}   # of a significand


def _experts(gen, kind, e, k, n, group, dtype):
    q = torch.randint(-2 ** 31, 2 ** 31 - 1, (e, k // 16, 2 * n), dtype=torch.int32, device=DEV, generator=gen)
    z = None
    if kind == "mxfp4":
        s = torch.randint(117, 122, (e, k // 32, n), dtype=torch.uint8, device=DEV, generator=gen).view(torch.float8_e8m0fnu)
    else:
        s = (torch.rand((e, k // group, n), device=DEV, generator=gen) * 9e-3 + 1e-3).to(dtype)
    if kind == "uint4":
        z = torch.randint(-2 ** 31, 2 ** 31 - 1, (e, k // group, n // 8), dtype=torch.int32, device=DEV, generator=gen)
    return q, s, z


# blocks of 8, 16 and 32 slots; few strips (workgroups of eight wavefronts) and many (of four)
@pytest.mark.gpu
@pytest.mark.parametrize("kind,group,dtype", [(k, g, d) for d in (torch.float16, torch.bfloat16) for g in (128, 64, 32)
                                              for k in ("uint4b8", "uint4")] + [("mxfp4", 32, torch.bfloat16)])
@pytest.mark.parametrize("tokens", [7, 24, 56])
@pytest.mark.parametrize("k,inter", [(384, 256), (2560, 4096)])
def test_layer(kind, group, dtype, tokens, k, inter):
    e, top_k = 4, 2
    gen = torch.Generator(device=DEV).manual_seed(tokens + k)
    w1, s1, z1 = _experts(gen, kind, e, k, 2 * inter, group, dtype)
    w2, s2, z2 = _experts(gen, kind, e, inter, k, group, dtype)
    bias1 = (torch.randn((e, 2 * inter), device=DEV, generator=gen) * 0.1).to(dtype)
    x = torch.randn((tokens, k), device=DEV, generator=gen).to(dtype) * 0.1
    weights, ids = torch.topk(torch.softmax(torch.randn((tokens, e), device=DEV, generator=gen), dim=1), top_k, dim=1)
    wtype = {"uint4b8": scalar_types.uint4b8, "uint4": scalar_types.uint4, "mxfp4": scalar_types.float4_e2m1f}[kind]
    block = fused_moe.moe_block_size(tokens, top_k, e)
    routed = [_lib.load().sonar_moe_routed_gemm_applies(tokens * top_k, block, e, wtype.id, n_, k_, k_ // group)
              for n_, k_ in ((2 * inter, k), (k, inter))]
    assert routed == [1, 1] or block == 32   # (blocks of 32 are the mid-size kernel's in part)
    for activation, on_input in (("gelu", False), ("swigluoai", False), ("silu", False), ("silu", True)):
        def layer(**kw):
            return fused_moe.fused_marlin_moe(x, w1, w2, bias1, None, s1, s2, weights.contiguous(), ids.to(torch.int32), wtype.id, on_input,
                                              activation=activation, w1_zeros=z1, w2_zeros=z2, **kw)
        got, want = layer(), layer(activation_func=fused_moe.apply_moe_activation)
        assert bool(torch.isfinite(want).all())
        if activation == "silu" or block == 32:   # (the layer with sorted slots may have run in the mid-size kernel, which adds in its order)
            # a value between the GEMMs, and one of the result, may be rounded the other way: one unit of their type each
            error = (got.double() - want.double()).norm() / want.double().norm()
            assert error < 2 * 2.0 ** -BITS[dtype], error
        else:
            assert torch.equal(got, want), activation


def _both(ids, experts, block, top_k=1, k=128, n=128):
    """Rows of C from the routed and from the sorted call; 7.0 where neither writes."""
    lib = _lib.load()
    slots = ids.numel()
    gen = torch.Generator(device=DEV).manual_seed(slots + block)
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (experts, k * n // 8), dtype=torch.int32, device=DEV, generator=gen)
    s = (torch.rand((experts, n), device=DEV, generator=gen) * 9e-3 + 1e-3).to(torch.bfloat16)
    a = torch.randn((slots // top_k, k), device=DEV, generator=gen).to(torch.bfloat16)
    tw = torch.rand(slots, device=DEV, generator=gen)
    ids = ids.to(torch.int32).to(DEV).contiguous()
    c = [torch.full((slots, n), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    stream = torch.cuda.current_stream().cuda_stream
    args = (block, top_k, 1, experts, _lib.DTYPE_BF16, _lib.TYPE_UINT4B8, slots // top_k, n, k, 1)
    _lib.check(lib.sonar_moe_routed_gemm(a.data_ptr(), c[0].data_ptr(), w.data_ptr(), _lib.LAYOUT_GFX950, None, s.data_ptr(), None,
                                         ids.data_ptr(), tw.data_ptr(), *args, None, 0, 0.0, 0.0, None, stream))
    length = slots + experts * (block - 1)
    blocks = -(-length // block)
    sorted_ids, expert_ids, past, offsets = (torch.empty(v, dtype=torch.int32, device=DEV) for v in (length, blocks, 1, experts))
    _lib.check(lib.sonar_moe_align_block_size(ids.data_ptr(), slots, experts, block, sorted_ids.data_ptr(), length, expert_ids.data_ptr(),
                                              blocks, past.data_ptr(), None, offsets.data_ptr(), stream))
    _lib.check(lib.sonar_moe_wna16_marlin_gemm(
        a.data_ptr(), c[1].data_ptr(), w.data_ptr(), _lib.LAYOUT_GFX950, None, s.data_ptr(), None, None, None, None, 0, None, 0,
        sorted_ids.data_ptr(), length, expert_ids.data_ptr(), past.data_ptr(), tw.data_ptr(), *args, 1, 0, 1, stream))
    torch.cuda.synchronize()
    return c


@pytest.mark.gpu
@pytest.mark.parametrize("block", [8, 16, 32])
@pytest.mark.parametrize("slots", [1, 31, 63, 64, 65, 96, 127, 128])
def test_routings(block, slots):
    rng = torch.Generator().manual_seed(slots)
    for ids, experts in ((torch.randint(0, 5, (slots,), generator=rng), 5),                  # uneven, every expert
                         (torch.randint(-3, 12, (slots,), generator=rng), 7),                # some out of range on either side
                         (torch.full((slots,), 3), 4),                                       # one expert: several blocks of it
                         (torch.randint(0, 256, (slots,), generator=rng), 256),              # the most experts
                         (torch.full((slots,), -1), 3),                                      # nothing to do
                         (torch.arange(slots) % 2 * 254, 255)):
        got, want = _both(ids, experts, block)
        assert torch.equal(got, want), (ids, experts)
    if slots % 2 == 0:   # two slots a token, an expert twice for some
        got, want = _both(torch.randint(0, 3, (slots,), generator=rng), 3, block, top_k=2)
        assert torch.equal(got, want)


# global_num_experts below the experts held: the slots of the others are left out, as with more slots than this path takes
@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [6, 100, 200])
def test_fewer_experts_than_held(tokens):
    e, inter, k, dtype = 4, 128, 256, torch.bfloat16
    gen = torch.Generator(device=DEV).manual_seed(tokens)
    w1, s1, _ = _experts(gen, "uint4b8", e, k, 2 * inter, 128, dtype)
    w2, s2, _ = _experts(gen, "uint4b8", e, inter, k, 128, dtype)
    x = torch.randn((tokens, k), device=DEV, generator=gen).to(dtype) * 0.1
    ids = (torch.arange(tokens, device=DEV, dtype=torch.int32) % e).view(tokens, 1).contiguous()
    weights = torch.ones((tokens, 1), device=DEV)

    def layer(experts):   # row i of either GEMM lies at i * k, as 2 * inter == k
        return fused_moe.fused_marlin_moe(
            x, w1, w2, None, None, s1, s2, weights, ids, scalar_types.uint4b8.id, global_num_experts=experts,
            intermediate_cache13=torch.full((tokens * k,), 7.0, dtype=dtype, device=DEV))
    whole, part = layer(e), layer(e - 1)
    left_out = ids[:, 0] == e - 1
    assert bool((part[left_out] == 7.0).all()) and not bool((whole == 7.0).all(dim=1).any())
    assert bool((part[~left_out] != 7.0).any(dim=1).all())
    with pytest.raises(RuntimeError, match="out of range"):   # refused with any number of slots
        layer(8193)


@pytest.mark.parametrize("slots,block,experts,code,n,k,groups,want", [
    (128, 8, 256, _lib.TYPE_UINT4B8, 128, 128, 1, 1), (129, 8, 8, _lib.TYPE_UINT4B8, 128, 128, 1, 0),
    (128, 8, 257, _lib.TYPE_UINT4B8, 128, 128, 1, 0), (128, 48, 8, _lib.TYPE_UINT4B8, 128, 128, 1, 0),
    (16, 8, 8, _lib.TYPE_UINT8B128, 128, 128, 1, 0), (16, 8, 8, _lib.TYPE_FLOAT4_E2M1F, 128, 256, 8, 1),
    (16, 8, 8, _lib.TYPE_FLOAT4_E2M1F, 128, 256, 16, 0), (16, 8, 8, _lib.TYPE_UINT4, 128, 192, 3, 0),
    (0, 8, 8, _lib.TYPE_UINT4, 128, 128, 1, 0), (16, 8, 8, _lib.TYPE_UINT4, 96, 128, 1, 0)])
def test_which_calls(slots, block, experts, code, n, k, groups, want):
    lib = _lib.load()
    assert lib.sonar_moe_routed_gemm_applies(slots, block, experts, code, n, k, groups) == want
    if not want and slots:   # refused before anything is launched
        one = ctypes.c_int(5)
        assert lib.sonar_moe_routed_gemm(None, None, None, _lib.LAYOUT_GFX950, None, None, None, 16, None, block, 1, 0, experts,
                                         _lib.DTYPE_BF16, code, slots, n, k, groups, None, 0, 0.0, 0.0, ctypes.byref(one), None) != 0


# The same layers with sorted slots (another process, which takes the routing from the decode kernel): where that kernel forms the
# activation either way, silu_and_mul included, the bits are the same.  Blocks of 8, 16 and 32 slots.
@pytest.mark.gpu
def test_same_bits_with_sorted_slots():
    out = [subprocess.run([sys.executable, "-u", "-m", "tests.test_gpu_moe_routed"], cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                          capture_output=True, text=True, env=dict(os.environ, **env), timeout=110)
           for env in ({}, {"SONAR_MARLIN_NO_MOE_ROUTED": "1"})]
    assert all(o.returncode == 0 and o.stdout.strip().endswith("done") for o in out), [o.stdout[-500:] + o.stderr[-1500:] for o in out]
    assert out[0].stdout == out[1].stdout


def _digests() -> None:
    routed = 0 if os.environ.get("SONAR_MARLIN_NO_MOE_ROUTED") else 1
    e, top_k, k, inter, group = 8, 2, 512, 2048, 32
    for kind, dtype in (("uint4b8", torch.float16), ("uint4", torch.bfloat16), ("mxfp4", torch.bfloat16)):
        for tokens, block in ((20, 8), (48, 16), (64, 32)):
            gen = torch.Generator(device=DEV).manual_seed(tokens)
            w1, s1, z1 = _experts(gen, kind, e, k, 2 * inter, group, dtype)
            w2, s2, z2 = _experts(gen, kind, e, inter, k, group, dtype)
            x = torch.randn((tokens, k), device=DEV, generator=gen).to(dtype) * 0.1
            weights, ids = torch.topk(torch.softmax(torch.randn((tokens, e), device=DEV, generator=gen), dim=1), top_k, dim=1)
            wtype = {"uint4b8": scalar_types.uint4b8, "uint4": scalar_types.uint4, "mxfp4": scalar_types.float4_e2m1f}[kind]
            assert fused_moe.moe_block_size(tokens, top_k, e) == block
            for n_, k_ in ((2 * inter, k), (k, inter)):
                assert _lib.load().sonar_moe_routed_gemm_applies(tokens * top_k, block, e, wtype.id, n_, k_, k_ // group) == routed
            rows = tokens * top_k
            for activation in ("silu", "swigluoai"):
                cache13 = torch.full((rows * 2 * inter,), -7.0, dtype=dtype, device=DEV)
                out = fused_moe.fused_marlin_moe(x, w1, w2, None, None, s1, s2, weights.contiguous(), ids.to(torch.int32), wtype.id,
                                                 activation=activation, w1_zeros=z1, w2_zeros=z2, intermediate_cache13=cache13)
                assert bool(torch.isfinite(out).all())
                # (rounds of workgroups on 256 compute units)
                if torch.cuda.get_device_properties(0).multi_processor_count == 256:
                    assert bool((cache13[rows * k:] == -7.0).all())   # no gate and up rows: the kernel formed the activation
                    assert _lib.load().sonar_marlin_last_grouped_kernel() == _lib.GROUPED_DECODE
                print(kind, tokens, activation, hashlib.sha256(out.view(torch.uint8).cpu().numpy().tobytes()).hexdigest()[:16], flush=True)


if __name__ == "__main__":
    _digests()
    print("done", flush=True)
