"""Calls of 17 to a few hundred rows on 4-bit integer weights with one group or groups of 128 rows or more keep their weights
exact: the matrix cores take the integers, and scales and zero points go into fp32 sums.  The error against the
product in 64 bits is then the output's own rounding.

Bound: independent errors add in squares, so 1.05 times the rounding error of the output leaves room for another of
0.32 of it.  fp32 sums add less than 0.02 of it here; rounding each scaled weight to 16 bits adds 0.8 (bfloat16: 1.3e-3 beside
1.65e-3; float16 the same in eighths), which gives 1.28."""
from __future__ import annotations

import os
import subprocess
import sys

import pytest
import torch

from sonar_amd import marlin_utils as mu
from sonar_amd import ops
from sonar_amd.scalar_type import scalar_types

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _call(m, k, n, group, dtype, zero_points, mean, columns):
    gen = torch.Generator(device=DEV).manual_seed(m + k + n)
    groups = 1 if group == -1 else k // group
    q = torch.randint(0, 16, (k, n), device=DEV, generator=gen, dtype=torch.int32)
    s = (torch.rand((groups, n), device=DEV, generator=gen) * 9e-3 + 1e-3).to(dtype)
    z = torch.randint(3, 13, (groups, n), device=DEV, generator=gen, dtype=torch.int32)
    a = (torch.randn((m, k), device=DEV, generator=gen) + mean).to(dtype)
    packed = q.view(k // 8, 8, n)[:, 0].clone()
    for t in range(1, 8):
        packed |= q.view(k // 8, 8, n)[:, t] << (4 * t)
    empty = torch.empty(0, dtype=torch.int32, device=DEV)
    weight = ops.gptq_marlin_repack(packed, empty, k, n, 4)
    scales = mu.marlin_permute_scales(s, k, n, group)
    zeros = mu.marlin_zero_points(z, groups, n, 4) if zero_points else empty
    out = mu.apply_gptq_marlin_linear(a, weight, scales, zeros, empty, empty, mu.marlin_make_workspace_new(torch.device(DEV)),
                                      scalar_types.uint4 if zero_points else scalar_types.uint4b8, n, k, True)
    pick = torch.arange(0, n, max(1, n // columns), device=DEV)
    rows = k // groups
    zero = z[:, pick].repeat_interleave(rows, 0).double() if zero_points else 8.0
    exact_w = (q[:, pick].double() - zero) * s[:, pick].repeat_interleave(rows, 0).double()
    return out[:, pick].double().cpu(), a.double().cpu() @ exact_w.cpu()


# pieces of strips and whole strips, one to many row tiles, K split over workgroups, ranges of unequal length and empty ones,
# a last tile of one row, an odd last strip
@pytest.mark.parametrize("m,k,n,group", [
    (17, 1024, 1024, 128), (33, 128, 192, -1), (64, 4096, 4096, 128), (64, 4096, 14336, 128), (49, 1152, 6208, 128), (63, 8192, 2048, 256),
    (128, 4096, 6144, 128), (200, 4096, 6144, 128), (113, 2048, 4160, -1), (64, 14336, 4096, -1), (256, 4096, 4096, 512), (24, 3072, 16384, 1024),
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("zero_points", [False, True])
def test_error_is_the_rounding_of_the_output(m, k, n, group, dtype, zero_points):
    _check(m, k, n, group, dtype, zero_points)


# tiles of every height, with K in one piece and in several; a child each, because the switch is read once per process
@pytest.mark.parametrize("row_blocks", ["2", "3", "4", "2,3", "3,8", "4,2"])
def test_tiles_of_every_height(row_blocks):
    out = subprocess.run([sys.executable, "-u", "-m", "tests.test_gpu_int4_precision"], cwd=ROOT, capture_output=True, text=True,
                         env=dict(os.environ, SONAR_MARLIN_MID_ROWS=row_blocks), timeout=110)
    assert out.returncode == 0 and "all shapes ok" in out.stdout, out.stdout[-1500:] + out.stderr[-1500:]


def _check(m, k, n, group, dtype, zero_points) -> None:
    for mean in (0.0, 0.5):
        got, exact = _call(m, k, n, group, dtype, zero_points, mean, 128)
        rounding = (exact.to(dtype).double() - exact).norm()
        assert (got - exact).norm() <= 1.05 * rounding, (mean, float((got - exact).norm() / rounding))


def main() -> None:
    rows = 16 * int(os.environ["SONAR_MARLIN_MID_ROWS"].split(",")[0])
    # one unit of K for four ranges; ranges of 6, 6, 6 and 0 steps, of 10, 10, 10 and 8, of 4, 4, 4 and 0; row tiles of one row
    for m, k, n, group in ((1, 128, 64, -1), (rows, 1152, 192, 128), (rows + 1, 2432, 448, 128), (2 * rows - 1, 768, 1088, 256),
                           (5 * rows + 3, 4096, 128, 512), (rows - 3, 1920, 320, -1)):
        for dtype in (torch.float16, torch.bfloat16):
            for zero_points in (False, True):
                print(m, k, n, group, dtype, zero_points, flush=True)
                _check(m, k, n, group, dtype, zero_points)
    print("all shapes ok", flush=True)


if __name__ == "__main__":
    main()
