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

# tokens, experts, K, N and slots of a block (top 2): half a round to a round of workgroups with blocks of 32, a quarter and more
# with 48; 64 rows and less an expert, and 100 (two blocks)
SHAPES = [(42, 4, 384, 4160, 32), (80, 4, 256, 2112, 48), (70, 3, 128, 2880, 48), (100, 4, 640, 320, 64), (200, 4, 128, 192, 64)]


@pytest.mark.parametrize("m,e,k,n,slots", SHAPES)
@pytest.mark.parametrize("group", [-1, 128])
@pytest.mark.parametrize("dtype,zp", [("fp16", False), ("fp16", True), ("bf16", False), ("bf16", True)])
def test_integer_codes(m, e, k, n, slots, group, dtype, zp):
    tm.test_moe_gemm_within_tolerance((m, e, 2, k, n, group, dtype, zp, False, zp, slots, not zp))


@pytest.mark.parametrize("m,e,k,n,slots", SHAPES)
def test_act_order(m, e, k, n, slots):
    if k > 128:
        tm.test_moe_gemm_within_tolerance((m, e, 2, k, n, 128, "bf16", False, True, True, slots, True))


# an expert with no rows, one with a single block, one with many: the routing of `route` over more experts than tokens reach
@pytest.mark.parametrize("slots", [48, 64])
def test_uneven_routing(slots):
    tm.test_moe_gemm_within_tolerance((230, 8, 1, 256, 1088, 128, "bf16", True, False, False, slots, True))


# 25, 37 and 47 rows an expert are blocks of 32, 48 and 64 slots
@pytest.mark.parametrize("tokens", [100, 150, 190])
@pytest.mark.parametrize("k,n", [(192, 4160), (1152, 2112)])
def test_mxfp4(tokens, k, n):
    tm.test_full_size_grouped_gemm_agrees_with_dense_rows(tokens, k, n, "mxfp4")


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
