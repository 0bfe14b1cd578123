"""Rows of results of the W4A8 kernel of gemm_a8_block.hip leave through LDS as 16-byte pieces: a matrix C that is aligned to
its elements only, ragged last tiles of rows and strips, and nothing written around C."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import marlin_oracle as mo
from sonar_amd import _lib
from tests.gpu_util import DEV, dtype_code, host_f32, ptr, stream
from tests.test_gpu_a8 import A8Layer

pytestmark = pytest.mark.gpu


# 17 to 64 rows: ranges of K summed in LDS; from 1000 rows: one wavefront a strip of 128 or 96 rows
@pytest.mark.parametrize("m,n", [(33, 320), (64, 1088), (1025, 1088), (1024, 2112)])
@pytest.mark.parametrize("offset", [0, 1, 4])
def test_rows_of_an_unaligned_result(m, n, offset):
    k, guard = 256, 64
    layer = A8Layer(7, k, n, 128, "fp16", False, "int8", bias=True)
    a_q, a_s = mo.per_token_quant_int8(np.random.default_rng(m).standard_normal((m, k)).astype(np.float32))
    a_s = (a_s * layer.factor).astype(np.float32)
    a, scales = torch.from_numpy(a_q).to(DEV), torch.from_numpy(a_s.reshape(-1)).to(DEV)
    whole = torch.full((m * n + 2 * guard,), -7.0, dtype=torch.float16, device=DEV)
    c = whole[guard + offset:guard + offset + m * n]
    lib = _lib.load()
    nbytes = lib.sonar_marlin_gemm_a8_scratch_bytes(m, n, k, layer.groups)
    scratch = torch.empty(max(nbytes, 16), dtype=torch.uint8, device=DEV)
    _lib.check(lib.sonar_marlin_gemm_a8(
        ptr(a), k, _lib.ADTYPE_INT8, ptr(c), ptr(layer.native), _lib.LAYOUT_GFX950, ptr(layer.dev_bias),
        ptr(layer.dev_scales), ptr(scales), None, ptr(scratch), scratch.numel(), dtype_code("fp16"), layer.b_type, m, n, k,
        layer.groups, stream()))
    want = mo.gemm_w4a8_int8(a_q, a_s, layer.q, 128, layer.scales, "fp16", None, layer.bias32)
    assert np.array_equal(host_f32(c).reshape(m, n), want)
    assert bool((whole[:guard + offset] == -7.0).all()) and bool((whole[guard + offset + m * n:] == -7.0).all())
