"""Launches of the wide tile kernel with both tile sizes: every form, dense (the kernel that would take calls of this size is
switched off, in a child process) and grouped, where the routing leaves 256-row and 128-row tiles."""
from __future__ import annotations

import os
import subprocess
import sys

import pytest

from tests import gpu_util as gu
from tests import test_gpu_moe as tm
from tests import test_gpu_parity as tp

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
def test_dense_forms(dtype):
    out = subprocess.run([sys.executable, "-u", "-m", "tests.test_gpu_two_tile_sizes", dtype], cwd=ROOT, capture_output=True,
                         text=True, env=dict(os.environ, SONAR_MARLIN_NO_MID="1"), timeout=110)
    assert out.returncode == 0 and "all forms ok" in out.stdout, out.stdout[-1500:] + out.stderr[-1500:]


def _dense(dtype: str) -> None:
    # 9 x 29 tiles: 256 as they are, five halved, of which some have no rows (52 in the last row tile)
    m, k, n = 2100, 192, 7360
    for g, zp in ((64, False), (64, True), (32, False), (32, True), (-1, True)):
        tp.test_wide_tile_kernel_forms_within_tolerance(gu, dtype, m, k, n, g, zp, zp)
        print(g, zp, "ok", flush=True)
    tp.test_w8a16_dequant_bit_exact_and_gemm_within_tolerance(gu, dtype, m, k, n, 64, False, True)
    tp.test_fp8_weights_dequant_bit_exact_and_gemm_within_tolerance(gu, dtype, m, k, n, -1, False)
    if dtype == "bf16":
        tp.test_mxfp4_weights_dequant_bit_exact_and_gemm_within_tolerance(gu, m, k, n, True)
    # 12 x 32 tiles, 128 halved, the last row tile with one row
    tp.test_wide_tile_kernel_forms_within_tolerance(gu, dtype, 2817, 128, 8192, 128, False, False)


# three experts of eleven or twelve blocks: 27 or 28 row tiles of 256 rows are too many for one round of tiles
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("g,zp", [(64, False), (64, True), (32, False), (32, True), (-1, False)])
def test_grouped_forms_on_integer_codes(dtype, g, zp):
    tm.test_moe_gemm_within_tolerance((1100, 3, 2, 192, 7424, g, dtype, zp, False, zp, 64, True))


@pytest.mark.parametrize("wtype", ["uint8b128", "fp8", "uint8b128/fp16", "fp8/fp16", "mxfp4", "uint4b8", "uint4b8/fp16"])
def test_grouped_forms_of_other_codes(wtype):
    tm.test_full_size_grouped_gemm_agrees_with_dense_rows(2300, 640, 4352, wtype)


# K of 16 steps or more in whole passes: tiles of both sizes cut along K, and their partial tiles added
@pytest.mark.parametrize("tokens,k,n", [(640, 4096, 2048), (1100, 14336, 1024), (2100, 4096, 1024)])
def test_grouped_tiles_cut_along_k(tokens, k, n):
    tm.test_full_size_grouped_gemm_agrees_with_dense_rows(tokens, k, n, "uint4b8")


if __name__ == "__main__":
    _dense(sys.argv[1])
    print("all forms ok", flush=True)
