"""Groups of 32 and 64 rows, and MXFP4, with blocks of 32, 48 and 64 slots in the grouped decode kernel: two blocks of 16 rows
share a unit's two or four sets of scales.  Workgroups of eight wavefronts (few strips) and of four (more (block, strip) pairs
than compute units); more wavefronts than units (K = 128); and K = 192, which is no whole number of units, in the general
kernel.  Tolerances are those of the grouped GEMM against the oracle, or against the dense call."""
from __future__ import annotations

import pytest

from tests import test_gpu_moe as tm

pytestmark = pytest.mark.gpu

FORMS = [(dtype, zp, group) for dtype in ("fp16", "bf16") for zp in (False, True) for group in (32, 64)]


@pytest.mark.parametrize("dtype,zp,group", FORMS)
@pytest.mark.parametrize("m,k,n,slots", [(40, 1280, 256, 32), (200, 256, 1024, 32), (60, 128, 128, 48), (120, 384, 320, 64)])
def test_integer_codes(m, k, n, slots, dtype, zp, group):
    tm.test_moe_gemm_within_tolerance((m, 4, 2, k, n, group, dtype, zp, False, zp, slots, True))


@pytest.mark.parametrize("dtype,zp,group", FORMS)
@pytest.mark.parametrize("slots", [32, 48])
def test_integer_codes_in_the_general_kernel(slots, dtype, zp, group):
    tm.test_moe_gemm_within_tolerance((40, 4, 2, 192, 128, group, dtype, zp, False, zp, slots, True))


# 25, 37 and 47 rows an expert are blocks of 32, 48 and 64 slots
@pytest.mark.parametrize("tokens", [100, 150, 190])
@pytest.mark.parametrize("k,n", [(512, 256), (1152, 4096), (192, 256)])
def test_mxfp4(tokens, k, n):
    tm.test_full_size_grouped_gemm_agrees_with_dense_rows(tokens, k, n, "mxfp4")


# sixteen experts in blocks of 64 slots, few strips: 1908 slots in the decode kernel, 2048 in the tile kernel
@pytest.mark.parametrize("dtype,zp,group", [("fp16", True, 128), ("bf16", False, 32)])
@pytest.mark.parametrize("tokens", [450, 520])
def test_sixteen_experts(tokens, dtype, zp, group):
    tm.test_moe_gemm_within_tolerance((tokens, 16, 2, 384, 192, group, dtype, zp, False, zp, 64, True))
