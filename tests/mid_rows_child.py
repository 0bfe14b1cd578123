"""Child process of test_gpu_mid_rows: with SONAR_MARLIN_MID_ROWS set (read once per process) every
dense call that the kernel of gemm_mid.hip can run goes to its tiles of that many row blocks ("rows,splits": with K
split over workgroups as well), here at the
edges of tiles, strips and K ranges, for every weight format, against the oracle."""
from __future__ import annotations

import os
import sys

import torch

from oracle import marlin_oracle as mo
from tests import gpu_util as gu
from tests import test_gpu_parity as tp


def int4(m, k, n, g, dtype, zp, bias) -> None:
    layer = gu.DeviceLayer(5 + m, k, n, g, dtype, zero_points=zp, bias=bias)
    a32 = mo.make_activations(m + 1, m, k, dtype, std=0.5)
    c = layer.gemm(gu.dev_bits16(a32, dtype), m)
    torch.cuda.synchronize()
    ok, max_err, max_ref = mo.gemm_tolerance_ok(gu.host_f32(c), mo.gemm_reference(a32, layer.w_ref, layer.bias32))
    if not ok:
        print("int4", m, k, n, g, dtype, zp, bias, f"FAILED max_err={max_err} max_ref={max_ref}", flush=True)
        sys.exit(1)


def main() -> None:
    rows = 16 * int(os.environ["SONAR_MARLIN_MID_ROWS"].split(",")[0])
    # one step of K for four ranges; an odd last strip; a last tile of one row; ranges of unequal length; many tiles;
    # ranges of 6 and 7 steps (the longer ring of a single row block)
    shapes = [(1, 64, 64), (rows, 320, 192), (rows + 1, 1344, 448), (2 * rows - 1, 512, 1088), (5 * rows + 3, 1024, 128), (rows - 3, 3136, 192)]
    for i, (m, k, n) in enumerate(shapes):
        for dtype in ("fp16", "bf16"):
            for g in (-1, 32, 64) + ((256,) if k % 256 == 0 and k > 256 else ()):
                if 0 < g < k or g == -1:
                    int4(m, k, n, g, dtype, False, i % 2 == 0)
                    int4(m, k, n, g, dtype, True, i % 2 == 1)
                    tp.test_w8a16_dequant_bit_exact_and_gemm_within_tolerance(gu, dtype, m, k, n, g, False, i % 2 == 0)
            for g in (-1, 32) + ((128,) if k % 128 == 0 and k > 128 else ()):
                if 0 < g < k or g == -1:
                    tp.test_fp8_weights_dequant_bit_exact_and_gemm_within_tolerance(gu, dtype, m, k, n, g, i % 2 == 1)
            tp.test_nvfp4_weights_dequant_bit_exact_and_gemm_within_tolerance(gu, m, k, n, i % 2 == 0, dtype)
        tp.test_mxfp4_weights_dequant_bit_exact_and_gemm_within_tolerance(gu, m, k, n, i % 2 == 1)
        print("shape", m, k, n, "ok", flush=True)
    tp.test_gemm_row_strided_activations(gu, *[(33, 512, 256)][0])
    print("all shapes ok", flush=True)


if __name__ == "__main__":
    main()
