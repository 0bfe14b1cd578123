"""K of every number of steps modulo four in the wide tile kernel, whose loop is passes of four steps that end early: one to
seven steps, and 45, on tiles of 256 and 128 rows, dense and grouped.  (The kernel that takes calls of this size is switched
off, in a child process, because the switches are read once per process.)"""
from __future__ import annotations

import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STEPS = (1, 2, 3, 4, 5, 6, 7, 45)


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
def test_every_tail_of_the_wide_kernel(dtype):
    out = subprocess.run([sys.executable, "-u", "-m", "tests.test_gpu_k_tails", dtype], cwd=ROOT, capture_output=True,
                         text=True, env=dict(os.environ, SONAR_MARLIN_NO_MID="1"), timeout=110)
    assert out.returncode == 0 and "all tails ok" in out.stdout, out.stdout[-1500:] + out.stderr[-1500:]


def _tails(dtype: str) -> None:
    from tests import gpu_util as gu
    from tests import test_gpu_moe as tm
    from tests import test_gpu_ops as to
    from tests import test_gpu_parity as tp
    for steps in STEPS:
        k = 64 * steps
        for g in (-1, 64, 32):
            for zp in (False, True):
                tp.test_wide_tile_kernel_forms_within_tolerance(gu, dtype, 600, k, 832, g, zp, not zp)      # 128-row tiles
        tp.test_wide_tile_kernel_forms_within_tolerance(gu, dtype, 2100, k, 4160, 64, steps % 2 == 0, False)   # 256
        tp.test_w8a16_dequant_bit_exact_and_gemm_within_tolerance(gu, dtype, 600, k, 320, 64, False, False)
        for g in (-1, 32):
            tp.test_fp8_weights_dequant_bit_exact_and_gemm_within_tolerance(gu, dtype, 600, k, 320, g, steps % 2 == 1)
        tp.test_nvfp4_weights_dequant_bit_exact_and_gemm_within_tolerance(gu, 600, k, 320, steps % 2 == 0, dtype)
        if dtype == "bf16":
            tp.test_mxfp4_weights_dequant_bit_exact_and_gemm_within_tolerance(gu, 600, k, 320, True)
        print("dense", k, "ok", flush=True)
        # more slots than the decode kernel takes: whole tiles and an expert's short end
        for g, zp in ((-1, False), (64, True), (32, False)):
            tm.test_moe_gemm_within_tolerance((900, 2, 2, k, 320, g, dtype, zp, False, not zp, 64, True))
        if dtype == "bf16":
            to.test_prepare_moe_mxfp4_layer_and_fused_marlin_moe((700, 2, 2, k, 128, True))
        print("grouped", k, "ok", flush=True)


if __name__ == "__main__":
    _tails(sys.argv[1])
    print("all tails ok", flush=True)
