"""Kernel forms that the other GPU cases do not launch, against the same oracles: forms that a faster kernel stands in
front of on most shapes (it is switched off for them, in a child process each, because the switches are read once per
process), and a few of the grouped kernels and of the kernel between decode and prefill."""
from __future__ import annotations

import os
import subprocess
import sys

import pytest

from tests import gpu_util as gu
from tests import test_gpu_a8 as ta
from tests import test_gpu_moe as tm
from tests import test_gpu_ops as to
from tests import test_gpu_parity as tp

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SWITCHES = ("SONAR_MARLIN_NO_MID=1", "SONAR_MARLIN_A8_SHAPE=0", "SONAR_MARLIN_NO_MOE_TILE=1", "SONAR_MARLIN_NO_MOE_MID=1")


@pytest.mark.parametrize("switch", SWITCHES)
def test_forms_behind_a_faster_kernel(switch):
    name, _, value = switch.partition("=")
    out = subprocess.run([sys.executable, "-u", "-m", "tests.test_gpu_kernel_forms", name], cwd=ROOT, capture_output=True,
                         text=True, env=dict(os.environ, **{name: value}), timeout=110)
    assert out.returncode == 0 and "all forms ok" in out.stdout, out.stdout[-1500:] + out.stderr[-1500:]


# K = 160 is no whole number of 128-row steps: blocks of rows of the first W4A8 kernel
@pytest.mark.parametrize("act", ["int8", "fp8"])
@pytest.mark.parametrize("group", [-1, 32])
@pytest.mark.parametrize("zp", [False, True])
def test_w4a8_on_k_of_no_whole_steps(act, group, zp):
    call = ta.test_w4a8_int8_gemm_bit_exact if act == "int8" else ta.test_w4a8_fp8_gemm_within_tolerance
    for dtype in ("fp16", "bf16"):
        call(160, 192, group, zp, dtype, zp, [40, 70])


# K = 96 is no whole number of 64-row steps: 8-bit codes and NVFP4 in the streaming kernels
@pytest.mark.parametrize("m", [5, 20, 40])
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
def test_few_rows_on_k_of_no_whole_steps(m, dtype):
    for g in (-1, 32):
        tp.test_w8a16_dequant_bit_exact_and_gemm_within_tolerance(gu, dtype, m, 96, 192, g, False, True)
        tp.test_fp8_weights_dequant_bit_exact_and_gemm_within_tolerance(gu, dtype, m, 96, 192, g, False)
    tp.test_nvfp4_weights_dequant_bit_exact_and_gemm_within_tolerance(gu, m, 96, 192, True, dtype)


# the longer ring of a single row block with a scale row a step
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
def test_fp8_decode_with_groups_on_many_strips(dtype):
    tp.test_fp8_weights_dequant_bit_exact_and_gemm_within_tolerance(gu, dtype, 9, 3072, 8320, 128, True)


@pytest.mark.parametrize("act", ["int8", "fp8"])
@pytest.mark.parametrize("block", [32, 48, 64])
@pytest.mark.parametrize("zp", [False, True])
def test_grouped_w4a8_with_groups(act, block, zp):
    ta.test_moe_w4a8_gemm(act, 2 * block, 256, 128, 3, 2, block, 64, zp, "bf16", zp, not zp)


# K = 192: the general grouped kernel with zero points; act-order through the gather
@pytest.mark.parametrize("block", [32, 48, 64])
@pytest.mark.parametrize("kind", ["zero_points", "act_order"])
def test_general_grouped_kernel_in_bf16(block, kind):
    if kind == "zero_points":
        tm.test_moe_gemm_within_tolerance((2 * block, 3, 2, 192, 128, 64, "bf16", True, False, True, block, True))
    else:
        tm.test_moe_gemm_within_tolerance((2 * block, 3, 2, 512, 128, 128, "bf16", False, True, False, block, True))


# 32-slot blocks (two blocks of rows) of fp8 and MXFP8 experts
def test_grouped_fp8_on_32_slot_blocks():
    to.test_prepare_fp8_moe_layer_and_fused_marlin_moe((40, 4, 2, 256, 128, "bf16", "channel"))
    to.test_prepare_mxfp8_moe_layer_and_fused_marlin_moe((40, 4, 2, 256, 128))


def _without_the_mid_kernel() -> None:
    for dtype in ("fp16", "bf16"):
        for m in (5, 20, 40, 64):
            for g in (-1, 32):
                tp.test_w8a16_dequant_bit_exact_and_gemm_within_tolerance(gu, dtype, m, 512, 192, g, False, m == 20)
                tp.test_fp8_weights_dequant_bit_exact_and_gemm_within_tolerance(gu, dtype, m, 512, 192, g, m == 40)
            tp.test_nvfp4_weights_dequant_bit_exact_and_gemm_within_tolerance(gu, m, 512, 192, m == 20, dtype)
            if dtype == "bf16":
                tp.test_mxfp4_weights_dequant_bit_exact_and_gemm_within_tolerance(gu, m, 512, 192, m == 20)
            for zp, act in ((False, False), (True, False), (False, True)):
                tp.test_marlin_gemm_within_tolerance(gu, dtype, m, 512, 192, 64, zp, act, m == 40)
        # 132 strips x 2 pairs of row blocks: the decode kernel with four wavefronts
        for g, zp in ((128, False), (-1, False), (128, True)):
            tp.test_marlin_gemm_within_tolerance(gu, dtype, 40, 512, 8448, g, zp, False, zp)
        print("streaming", dtype, "ok", flush=True)
        for case in tp.TILE_CASES:
            if case[3] == 32:
                tp.test_marlin_gemm_tiled_within_tolerance(gu, dtype, *case)
        for case in tp.WIDE_TILE_CASES:
            if case[3] == 32:
                tp.test_wide_tile_kernel_forms_within_tolerance(gu, dtype, *case)
        tp.test_wide_tile_kernel_forms_within_tolerance(gu, dtype, 600, 1216, 512, 32, True, True)
        print("tiles", dtype, "ok", flush=True)


def _without_the_w4a8_block_kernel() -> None:
    for dtype in ("fp16", "bf16"):
        for zp in (False, True):
            for group in (-1, 64, 128):   # N = 192: blocks of 16 rows; N = 256, more than 32 rows: tiles
                ta.test_w4a8_int8_gemm_bit_exact(512, 192, group, zp, dtype, zp, [40, 70])
                ta.test_w4a8_fp8_gemm_within_tolerance(512, 192, group, zp, dtype, zp, [40, 70])
                ta.test_w4a8_int8_gemm_bit_exact(1024, 256, group, zp, dtype, not zp, [100, 257])
                ta.test_w4a8_fp8_gemm_within_tolerance(1024, 256, group, zp, dtype, not zp, [100, 257])
        print("w4a8", dtype, "ok", flush=True)


def _without_the_grouped_tile_kernel() -> None:
    # 64-slot blocks: four blocks of rows of the general grouped kernels
    to.test_prepare_fp8_moe_layer_and_fused_marlin_moe((110, 4, 2, 256, 128, "bf16", "channel"))
    to.test_prepare_mxfp8_moe_layer_and_fused_marlin_moe((110, 4, 2, 256, 128))
    to.test_prepare_nvfp4_moe_layer_and_fused_marlin_moe((110, 4, 2, 256, 128), "bf16")


def _without_the_grouped_mid_kernel() -> None:
    """Blocks of 32 slots and more of 4-bit codes that marlin_mid_gemm takes: in the kernels that the cases are named after."""
    from sonar_amd import _lib
    from tests import test_gpu_moe_small_groups as ts
    last = _lib.load().sonar_marlin_last_grouped_kernel

    def ran(kernel, call, *args):
        call(*args)
        assert last() == kernel, (call.__name__, args, last())
        print(call.__name__, args, "ok", flush=True)

    for case in [(700, 4, 2, 1024, 320, 128, "fp16", False, False, False, 64, True),      # K split in both tile sizes
                 (900, 3, 2, 2048, 256, 128, "bf16", True, False, True, 64, False),
                 (650, 2, 2, 1024, 256, 128, "fp16", False, True, False, 64, True),       # act-order: rows of A by slot
                 (1100, 2, 1, 128, 512, 128, "bf16", False, False, True, 64, False),
                 (600, 4, 2, 512, 256, 128, "fp16", True, False, True, 64, True),
                 (700, 4, 2, 512, 256, -1, "bf16", False, False, False, 64, True),
                 (700, 2, 2, 640, 256, 128, "fp16", False, False, True, 64, True)]:
        ran(_lib.GROUPED_TILE, tm.test_moe_gemm_within_tolerance, case)
    ran(_lib.GROUPED_TILE, tm.test_full_size_grouped_gemm_agrees_with_dense_rows, 700, 2048, 1024, "uint4b8/fp16")
    ran(_lib.GROUPED_TILE, tm.test_full_size_grouped_gemm_agrees_with_dense_rows, 700, 4096, 2048, "mxfp4")
    ran(_lib.GROUPED_TILE, tm.test_tile_kernel_with_expert_ids_that_are_not_grouped_by_expert, 128)
    ran(_lib.GROUPED_GENERAL, tm.test_full_size_grouped_gemm_agrees_with_dense_rows, 300, 512, 256, "mxfp4!")
    for dtype, zp in (("bf16", False), ("fp16", False), ("fp16", True), ("bf16", True)):
        ran(_lib.GROUPED_GENERAL, tm.test_moe_tiled_and_streaming_kernels_agree, dtype, zp, 128)
    for tokens in (100, 150, 190):
        ran(_lib.GROUPED_DECODE, ts.test_mxfp4, tokens, 1152, 4096)
    ran(_lib.GROUPED_DECODE, ts.test_sixteen_experts, 450, "fp16", True, 128)
    ran(_lib.GROUPED_TILE, ts.test_sixteen_experts, 520, "fp16", True, 128)
    for case in [(200, 4, 2, 256, 1024, 128, "bf16", True, False, False, 32, True),
                 (150, 4, 2, 256, 256, 128, "fp16", False, False, False, 48, True),
                 (120, 4, 2, 512, 1024, 128, "fp16", True, False, True, 64, True)]:
        ran(_lib.GROUPED_DECODE, tm.test_moe_gemm_within_tolerance, case)


if __name__ == "__main__":
    {"SONAR_MARLIN_NO_MID": _without_the_mid_kernel, "SONAR_MARLIN_A8_SHAPE": _without_the_w4a8_block_kernel,
     "SONAR_MARLIN_NO_MOE_TILE": _without_the_grouped_tile_kernel,
     "SONAR_MARLIN_NO_MOE_MID": _without_the_grouped_mid_kernel}[sys.argv[1]]()
    print("all forms ok", flush=True)
