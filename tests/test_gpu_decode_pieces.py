"""Strips of a decode launch in pieces of unequal length: the launch that is made, its results against the oracle, the
workspace afterwards, and the same with the pieces summed by the fix-up launch (a child process, because that switch is read
once per process)."""
from __future__ import annotations

import ctypes
import os
import subprocess
import sys

import pytest
import torch

from oracle import marlin_oracle as mo

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# m, k, n, group, dtype, zero points, pieces on 256 compute units.  The 8 units of 128 rows that a piece's wavefronts take at a
# time decide: more pieces than rounds are saved by; a prime number of units; a workgroup less than room; two and three blocks of rows.
CASES = [
    (1, 1024, 2432, 128, "bf16", False, 1),
    (8, 3328, 320, 128, "fp16", True, 4),       # 26 units: 6, 7, 6, 7
    (16, 10368, 1280, 128, "bf16", False, 8),   # 81 units
    (5, 5248, 5440, 64, "bf16", True, 3),       # 41 units, 85 strips: 255 workgroups
    (3, 7296, 5504, -1, "fp16", False, 2),      # 57 units, 86 strips: a third piece would be 258
    (12, 3712, 4096, 32, "fp16", False, 4),     # 29 units, 64 strips: every compute unit
    (32, 5504, 1664, -1, "bf16", False, None),  # 43 units in blocks of rows, where that kernel is chosen
    (48, 14208, 448, 128, "fp16", True, None),
]


@pytest.mark.parametrize("pieces", [2, 3, 4, 8])
def test_products_with_the_reciprocal_are_quotients(pieces):
    recip = 0xffffffff // pieces + 1
    top = [x for q in (1 << 16, 1 << 20, (1 << 28) // pieces) for x in range(q * pieces - 2, q * pieces + 2)]
    for x in list(range(1 << 12)) + top:
        assert (x * recip) >> 32 == x // pieces


def _check(m, k, n, group, dtype, zp, pieces):
    from sonar_amd import _lib
    from tests import gpu_util as gu
    layer = gu.DeviceLayer(3 + m, k, n, group, dtype, zero_points=zp, bias=m % 2 == 0)
    a32 = mo.make_activations(m + 5, m, k, dtype, std=0.5)
    a = gu.dev_bits16(a32, dtype)
    c = layer.gemm(a, m)
    torch.cuda.synchronize()
    launch = (ctypes.c_int32 * 4)()
    _lib.load().sonar_marlin_last_decode_launch(launch, 4)
    if pieces is not None and torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert launch[2] == pieces
    ok, max_err, max_ref = mo.gemm_tolerance_ok(gu.host_f32(c), mo.gemm_reference(a32, layer.w_ref, layer.bias32))
    assert ok, f"max_err={max_err} max_ref={max_ref}"
    assert int(layer.workspace.abs().sum().item()) == 0
    assert torch.equal(c.view(torch.int16), layer.gemm(a, m).view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=str)
def test_pieces_of_unequal_length(case):
    _check(*case)


@pytest.mark.gpu
def test_pieces_of_unequal_length_in_the_fixup_launch():
    env = dict(os.environ, SONAR_MARLIN_NO_INLINE_SUM="1")
    out = subprocess.run([sys.executable, "-u", "-m", "tests.test_gpu_decode_pieces"], cwd=ROOT, env=env,
                         capture_output=True, text=True, timeout=110)
    assert out.returncode == 0 and "all pieces ok" in out.stdout, out.stdout[-1500:] + out.stderr[-1500:]


if __name__ == "__main__":
    for one in CASES:
        print(one, flush=True)
        _check(*one)
    print("all pieces ok", flush=True)
