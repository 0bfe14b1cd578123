"""Groups of 192 rows, a multiple of 64 that is no power of two times 64: what the eight-wavefront tile kernel is left with,
dense and grouped, 4-bit and 8-bit integers.  Tolerances as in the tests that these cases go through; the grouped 8-bit call
against the product of the dequantised weights in 64 bits, from which it differs by fp32 sums and one rounding to the output
type (2^-9 of a value in bf16): within 1e-2 of the largest output, the tolerance of the other GEMM tests."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import marlin_oracle as mo
from sonar_amd import _lib
from tests import gpu_util as gu
from tests import test_gpu_moe as tm
from tests import test_gpu_parity as tp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("zp", [False, True])
def test_int4(dtype, zp):
    tp.test_wide_tile_kernel_forms_within_tolerance(gu, dtype, 300, 1152, 4160, 192, zp, zp)
    tm.test_moe_gemm_within_tolerance((700, 2, 2, 576, 320, 192, dtype, zp, False, zp, 64, True))


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
def test_uint8b128(dtype):
    tp.test_w8a16_dequant_bit_exact_and_gemm_within_tolerance(gu, dtype, 300, 1152, 4160, 192, False, False)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_uint8b128_experts(dtype):
    tokens, e, top_k, k, n, groups, bs = 700, 2, 1, 1152, 320, 6, 64
    lib = _lib.load()
    code = _lib.DTYPE_F16 if dtype == torch.float16 else _lib.DTYPE_BF16
    gen = torch.Generator(device=gu.DEV).manual_seed(3)
    native = torch.randint(-2 ** 31, 2 ** 31 - 1, (e, k * n // 4), dtype=torch.int32, device=gu.DEV, generator=gen)
    scales = (torch.rand((e, groups, n), device=gu.DEV, generator=gen) * 5e-4 + 1e-4).to(dtype)
    a = torch.randn((tokens, k), device=gu.DEV, generator=gen).to(dtype)
    topk_ids, _ = tm.route(5, tokens, e, top_k)
    sorted_ids, expert_ids, past = mo.moe_align_block_size(topk_ids, bs, e)
    sid, eid, npp = (gu.dev_i32(np.asarray(x, dtype=np.int32)) for x in (sorted_ids, expert_ids, [int(past[0])]))
    c = torch.zeros((tokens, n), dtype=dtype, device=gu.DEV)
    ws = torch.zeros(1024, dtype=torch.int32, device=gu.DEV)
    scr = torch.empty(max(lib.sonar_moe_marlin_gemm_scratch_bytes(sid.numel(), bs, n, k), 16), dtype=torch.uint8, device=gu.DEV)
    _lib.check(lib.sonar_moe_wna16_marlin_gemm(
        gu.ptr(a), gu.ptr(c), gu.ptr(native), _lib.LAYOUT_GFX950, None, gu.ptr(scales), None, None, None, gu.ptr(ws),
        ws.numel(), gu.ptr(scr), scr.numel(), gu.ptr(sid), sid.numel(), gu.ptr(eid), gu.ptr(npp), None, bs, top_k, 0, e, code,
        _lib.TYPE_UINT8B128, tokens, n, k, groups, 1, 0, 1, gu.stream()))
    for ex in range(e):
        rows = torch.from_numpy(np.nonzero(topk_ids[:, 0] == ex)[0]).to(gu.DEV)
        w = torch.empty((k, n), dtype=dtype, device=gu.DEV)
        _lib.check(lib.sonar_marlin_dequant(gu.ptr(native[ex]), _lib.LAYOUT_GFX950, gu.ptr(scales[ex]), None, None, gu.ptr(w),
                                            code, _lib.TYPE_UINT8B128, n, k, groups, 1, gu.stream()))
        want = a[rows].double() @ w.double()
        err = float((c[rows].double() - want).abs().max())
        assert rows.numel() > 256 and err <= 1e-2 * float(want.abs().max()), (ex, err)
