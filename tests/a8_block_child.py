"""Child process of test_gpu_a8_block: with SONAR_MARLIN_A8_SHAPE set (read once per process) every W4A8 call
that the kernel of gemm_a8_block.hip can run goes to that tile, here at the edges of tiles, strips, steps and
K ranges, for every form of scales and zero points, against the oracle."""
from __future__ import annotations

import os

from tests import test_gpu_a8 as ta


def main() -> None:
    rows = 32 * int(os.environ["SONAR_MARLIN_A8_SHAPE"].split(",")[0])
    # one step of K; fewer steps than ranges; ranges of unequal length; an odd last strip; a last tile of one row
    shapes = [(128, 64, [1, rows]), (384, 192, [rows + 1]), (1152, 320, [2 * rows - 1]), (1664, 1088, [3 * rows + 5])]
    for i, (k, n, ms) in enumerate(shapes):
        for group in (-1, 32, 64, 128):
            if group >= k:
                continue
            for zp in (False, True):
                dtype = "fp16" if (i + zp) % 2 else "bf16"
                ta.test_w4a8_int8_gemm_bit_exact(k, n, group, zp, dtype, (i + zp) % 2 == 0, ms)
                if group != 32:
                    ta.test_w4a8_fp8_gemm_within_tolerance(k, n, group, zp, dtype, (i + zp) % 2 == 0, ms)
        print("shape", k, n, ms, "ok", flush=True)
    print("all shapes ok", flush=True)


if __name__ == "__main__":
    main()
