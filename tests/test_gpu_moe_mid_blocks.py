"""Grouped calls in marlin_mid_gemm: blocks of 32, 48 and 64 slots in every form (4-bit integers with and without zero points,
one group or groups of 128 rows, MXFP4), an odd last strip, K of fewer steps than a workgroup has ranges, experts without rows and
with several blocks, and act-order experts (rows of A by slot).  Tolerances are those of the grouped GEMM against the oracle, or
against the dense call."""
from __future__ import annotations

import pytest
import torch

from oracle import marlin_oracle as mo
from sonar_amd import _lib
from tests import gpu_util as gu
from tests import test_gpu_moe as tm

pytestmark = pytest.mark.gpu

# tokens, experts, K, N and slots of a block (top 2): half a round to a round of workgroups on 256 compute units; most experts are
# one block, and in the last shape two
SHAPES = [(42, 4, 384, 4160, 32), (160, 8, 256, 2112, 48), (120, 6, 128, 2880, 48), (200, 8, 640, 2112, 64), (200, 4, 128, 192, 64)]


def _ran(call, *args):
    call(*args)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert _lib.load().sonar_marlin_last_grouped_kernel() == _lib.GROUPED_MID


@pytest.mark.parametrize("m,e,k,n,slots", SHAPES)
@pytest.mark.parametrize("group", [-1, 128])
@pytest.mark.parametrize("dtype,zp", [("fp16", False), ("fp16", True), ("bf16", False), ("bf16", True)])
def test_integer_codes(m, e, k, n, slots, group, dtype, zp):
    _ran(tm.test_moe_gemm_within_tolerance, (m, e, 2, k, n, group, dtype, zp, False, zp, slots, not zp))


@pytest.mark.parametrize("m,e,k,n,slots", SHAPES)
def test_act_order(m, e, k, n, slots):
    if k > 128:
        _ran(tm.test_moe_gemm_within_tolerance, (m, e, 2, k, n, 128, "bf16", False, True, True, slots, True))


# an expert with no rows, one with a single block, one with many: the routing of `route` over more experts than tokens reach
@pytest.mark.parametrize("slots", [48, 64])
def test_uneven_routing(slots):
    _ran(tm.test_moe_gemm_within_tolerance, (230, 8, 1, 256, 2112, 128, "bf16", True, False, False, slots, True))


# 25, 37 and 47 rows an expert are blocks of 32, 48 and 64 slots; K of an odd number of steps, and of whole units
@pytest.mark.parametrize("tokens", [100, 150, 190])
@pytest.mark.parametrize("k,n", [(192, 2112), (1152, 2112)])
def test_mxfp4(tokens, k, n):
    _ran(tm.test_full_size_grouped_gemm_agrees_with_dense_rows, tokens, k, n, "mxfp4")


# more than a round of workgroups of two strips: four strips a workgroup, the last of which has one, two and three of its own; K of an odd
# number of units and of fewer steps in the second range; experts with second blocks
FOUR = [(16, 200, 640, 4160, 32), (16, 296, 640, 2240, 48), (16, 400, 512, 2176, 64), (16, 400, 1152, 3136, 64), (8, 240, 1664, 1984, 64)]


@pytest.mark.parametrize("e,m,k,n,slots", FOUR)
@pytest.mark.parametrize("dtype,zp,group", [("fp16", False, 128), ("fp16", True, -1), ("bf16", True, 128), ("bf16", False, -1)])
def test_four_strips(e, m, k, n, slots, dtype, zp, group):
    _ran(tm.test_moe_gemm_within_tolerance, (m, e, 2, k, n, group, dtype, zp, False, zp, slots, not zp))


def test_four_strips_act_order():
    _ran(tm.test_moe_gemm_within_tolerance, (400, 16, 2, 640, 2240, 128, "bf16", False, True, True, 64, True))


@pytest.mark.parametrize("tokens,n", [(100, 8256), (150, 5184), (190, 5248)])
@pytest.mark.parametrize("k", [640, 1152])
def test_four_strips_mxfp4(tokens, k, n):
    _ran(tm.test_full_size_grouped_gemm_agrees_with_dense_rows, tokens, k, n, "mxfp4")


# the gated activation where the ranges meet: the bits of the layer whose activation is a launch of its own.  Blocks of 48 and 64 slots, of
# 32 with less than a round; two and four strips a workgroup, an odd number of strips in a half, experts with second blocks
@pytest.mark.parametrize("kind,group,dtype", [("uint4b8", 128, torch.float16), ("uint4", 128, torch.bfloat16), ("mxfp4", 32, torch.bfloat16)])
@pytest.mark.parametrize("e,tokens,k,inter", [(8, 92, 512, 1344), (8, 150, 512, 960), (8, 200, 1152, 832), (16, 296, 640, 1344), (16, 400, 1152, 1600),
                                              (4, 250, 640, 1088)])
def test_gated_activation(e, tokens, k, inter, kind, group, dtype):
    from sonar_amd import fused_moe
    from sonar_amd.scalar_type import scalar_types
    from tests.test_gpu_moe_routed import _experts
    gen = torch.Generator(device=gu.DEV).manual_seed(tokens + k)
    w1, s1, z1 = _experts(gen, kind, e, k, 2 * inter, group, dtype)
    w2, s2, z2 = _experts(gen, kind, e, inter, k, min(group, 64), dtype)
    bias1 = (torch.randn((e, 2 * inter), device=gu.DEV, generator=gen) * 0.1).to(dtype)
    x = torch.randn((tokens, k), device=gu.DEV, generator=gen).to(dtype) * 0.1
    weights, ids = torch.topk(torch.softmax(torch.randn((tokens, e), device=gu.DEV, generator=gen), dim=1), 2, dim=1)
    wtype = {"uint4b8": scalar_types.uint4b8, "uint4": scalar_types.uint4, "mxfp4": scalar_types.float4_e2m1f}[kind]
    for activation, on_input in (("swigluoai", False), ("silu", False), ("silu", True)):
        def layer(**kw):
            return fused_moe.fused_marlin_moe(x, w1, w2, bias1, None, s1, s2, weights.contiguous(), ids.to(torch.int32), wtype.id, on_input,
                                              activation=activation, w1_zeros=z1, w2_zeros=z2, **kw)
        got, want = layer(), layer(activation_func=fused_moe.apply_moe_activation)
        assert bool(torch.isfinite(want).all()) and torch.equal(got, want), activation


# the edges of the rule: experts, tokens (top 2), K, N, slots of a block, zero points, and the kernel
RULE = [(8, 72, 128, 2048, 32, False, "DECODE"), (8, 100, 128, 2048, 32, False, "MID"), (8, 100, 128, 2112, 32, False, "MID"), (8, 100, 128, 4096, 32, True, "DECODE"),
        (8, 120, 128, 1920, 48, True, "DECODE"), (8, 120, 128, 1984, 48, False, "MID"), (8, 120, 128, 8320, 48, False, "MID"),
        (8, 180, 128, 2048, 48, False, "DECODE"),    # 45 slots an expert: nearly full blocks
        (8, 200, 128, 4096, 64, True, "MID"), (8, 200, 128, 4224, 64, True, "DECODE"), (8, 200, 128, 5248, 64, True, "MID"),
        (32, 800, 128, 1024, 64, False, "MID"), (32, 800, 128, 2048, 64, False, "TILE"),   # one round, and a short K in two
        (32, 830, 1152, 1216, 64, False, "MID"), (32, 896, 1152, 2048, 64, False, "TILE")]  # 1.25 rounds; 2 of more blocks than experts


@pytest.mark.parametrize("e,m,k,n,slots,zp,kernel", RULE)
def test_rule(e, m, k, n, slots, zp, kernel):
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("rounds of workgroups on 256 compute units")
    tm.test_moe_gemm_within_tolerance((m, e, 2, k, n, 128, "bf16", zp, False, False, slots, False))
    assert _lib.load().sonar_marlin_last_grouped_kernel() == getattr(_lib, "GROUPED_" + kernel)


# the kernel reads scales 16 bytes a lane; the others take them at any 4
@pytest.mark.parametrize("offset", [2, 4, 8])   # elements of two bytes
@pytest.mark.parametrize("zp", [False, True])
def test_scales_at_fewer_than_16_bytes(offset, zp):
    m, e, top_k, k, n, slots = 200, 8, 2, 256, 2112, 64
    ex = tm.Experts(9, e, k, n, 128, "fp16", zp)
    sorted_ids, expert_ids, past = mo.moe_align_block_size(tm.route(3, m, e, top_k)[0], slots, e)
    a32 = mo.make_activations(4, m, k, "fp16")
    want = ex.reference(a32, sorted_ids, expert_ids, int(past[0]), slots, top_k, m, None)
    room = torch.empty(ex.scales.numel() + offset, dtype=ex.scales.dtype, device=gu.DEV)
    moved = room[offset:].view(ex.scales.shape).copy_(ex.scales)
    for scales, kernel in ((ex.scales, _lib.GROUPED_MID), (moved, _lib.GROUPED_MID if offset == 8 else _lib.GROUPED_DECODE)):
        ex.scales = scales
        got = gu.host_f32(ex.gemm(gu.dev_bits16(a32, "fp16"), sorted_ids, expert_ids, int(past[0]), None, slots, top_k, m, False))
        assert _lib.load().sonar_marlin_last_grouped_kernel() == kernel
        ok, *worst = mo.gemm_tolerance_ok(got, want)
        assert ok, worst
