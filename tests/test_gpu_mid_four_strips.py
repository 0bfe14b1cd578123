"""Dense calls of 4-bit integers in 64-row tiles of four strips (gemm_mid.hip): more than a round of workgroups of two strips on 256
compute units; a last tile with one and three strips of its own, row tiles of one row and full, K in an odd number of units."""
from __future__ import annotations

import pytest
import torch

from oracle import marlin_oracle as mo
from tests import gpu_util as gu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("zp", [False, True])
@pytest.mark.parametrize("m,k,n,group", [(65, 640, 24640, 128), (128, 1408, 24768, -1), (97, 1152, 16576, 128)])
def test_against_the_oracle(m, k, n, group, zp, dtype):
    layer = gu.DeviceLayer(5 + m, k, n, group, dtype, zero_points=zp, bias=zp)
    a32 = mo.make_activations(m + 1, m, k, dtype, std=0.5)
    c = layer.gemm(gu.dev_bits16(a32, dtype), m)
    torch.cuda.synchronize()
    ok, max_err, max_ref = mo.gemm_tolerance_ok(gu.host_f32(c), mo.gemm_reference(a32, layer.w_ref, layer.bias32))
    assert ok, (max_err, max_ref)
