"""bfloat16 calls on 8-bit weights with one scale a column keep their weights exact, whichever kernel the estimates choose: every
code is a bfloat16 number, and the scale goes into the fp32 sums.  The error against the product in 64 bits is then the output's
own rounding.

Bound: independent errors add in squares, so 1.05 times the rounding error of the output leaves room for another of 0.32
of it.  fp32 sums add less than 0.05 of it here; scaled weights rounded to bfloat16 add 0.95 (measured: 1.38 to 1.41 times)."""
from __future__ import annotations

import os
import subprocess
import sys
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from sonar_amd import _lib
from sonar_amd import marlin_utils as mu
from sonar_amd import marlin_utils_fp8 as f8
from sonar_amd import ops
from sonar_amd.scalar_type import scalar_types

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# tiles of 128 rows, of 256 rows, of both sizes in one launch, cut along K; K of no whole pass of four steps; ragged last tiles
SHAPES = [(582, 1280, 6912), (808, 5248, 3072), (128, 8192, 8192), (2048, 4096, 4096), (3000, 1216, 5120), (2200, 3072, 7360),
          (1500, 14336, 1600), (4097, 512, 4160), (300, 4096, 4096)]


def _call(m, k, n, fp8, mean, bias):
    gen = torch.Generator(device=DEV).manual_seed(m + k + n)
    a = (torch.randn((m, k), device=DEV, generator=gen) + mean).bfloat16()
    b = torch.randn(n, device=DEV, generator=gen).bfloat16() if bias else None
    pick = torch.arange(0, n, max(1, n // 128), device=DEV)
    if fp8:
        weight = (torch.randn((n, k), device=DEV, generator=gen) * 64).to(torch.float8_e4m3fn)
        scale = (torch.rand(n, device=DEV, generator=gen) * 3e-4 + 1e-4).bfloat16()
        layer = SimpleNamespace(output_size_per_partition=n, input_size_per_partition=k, params_dtype=torch.bfloat16,
                                orig_dtype=torch.bfloat16, bias=None if b is None else b.clone(), weight=weight, weight_scale=scale.float())
        w = weight.float()[pick].double() * scale[pick, None].double()
        f8.prepare_fp8_layer_for_marlin(layer, size_k_first=False)
        out = f8.apply_fp8_marlin_linear(a, layer.weight, layer.weight_scale, layer.workspace, n, k, layer.bias)
    else:
        q = torch.randint(0, 256, (k, n), device=DEV, generator=gen, dtype=torch.int32)
        scale = (torch.rand((1, n), device=DEV, generator=gen) * 6e-4 + 6e-5).bfloat16()
        w = ((q[:, pick].double() - 128) * scale[:, pick].double()).t()
        packed = q.view(k // 4, 4, n)[:, 0].clone()
        for t in range(1, 4):
            packed |= q.view(k // 4, 4, n)[:, t] << (8 * t)
        empty = torch.empty(0, dtype=torch.int32, device=DEV)
        out = mu.apply_gptq_marlin_linear(a, ops.gptq_marlin_repack(packed, empty, k, n, 8), mu.marlin_permute_scales(scale, k, n, -1),
                                          empty, empty, empty, mu.marlin_make_workspace_new(torch.device(DEV)),
                                          scalar_types.uint8b128, n, k, True, bias=None if b is None else mu.marlin_permute_bias(b))
    exact = a.double().cpu() @ w.t().contiguous().cpu()
    return out[:, pick].double().cpu(), exact if b is None else exact + b[pick].double().cpu()


def _check(m, k, n, fp8):
    for mean, bias in ((0.0, False), (0.5, True)):
        got, exact = _call(m, k, n, fp8, mean, bias)
        rounding = (exact.bfloat16().double() - exact).norm()
        assert (got - exact).norm() <= 1.05 * rounding, (m, k, n, fp8, mean, float((got - exact).norm() / rounding))


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("m,k,n", SHAPES)
def test_error_is_the_rounding_of_the_output(m, k, n, fp8):
    _check(m, k, n, fp8)


def test_in_the_tile_kernel_alone():
    """A child process, because the switch is read once."""
    out = subprocess.run([sys.executable, "-u", "-m", "tests.test_gpu_8bit_precision"], cwd=ROOT, capture_output=True, text=True,
                         env=dict(os.environ, SONAR_MARLIN_NO_MID="1"), timeout=110)
    assert out.returncode == 0 and "all shapes ok" in out.stdout, out.stdout[-1500:] + out.stderr[-1500:]


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("tokens,k,n", [(700, 4096, 2048), (700, 640, 512), (2048, 2048, 1024), (300, 4096, 256)])
def test_experts(tokens, k, n, fp8):
    """A grouped call gives what dense calls of up to 16 rows of the same expert give, which keep the weights exact: only sums
    that fp32 leaves on the other side of a rounding step differ (fewer than one in a hundred: 0.35 of the rounding error)."""
    from oracle import marlin_oracle as mo
    from tests import gpu_util as gu
    from tests.test_gpu_moe import route
    e, top_k = 8, 2
    gen = torch.Generator(device=DEV).manual_seed(tokens + n)
    lib = _lib.load()
    b_type = _lib.TYPE_FLOAT8_E4M3FN if fp8 else _lib.TYPE_UINT8B128
    native = torch.randint(-2 ** 31, 2 ** 31 - 1, (e, k * n // 4), dtype=torch.int32, device=DEV, generator=gen)
    scales = torch.rand((e, 1, n), device=DEV, generator=gen) * 6e-4 + 6e-5
    scales = (scales * (2.0 ** 120 if fp8 else 1.0)).bfloat16()
    a = torch.randn((tokens, k), device=DEV, generator=gen).bfloat16()
    topk_ids, _ = route(tokens, tokens, e, top_k)
    sorted_ids, expert_ids, past = mo.moe_align_block_size(topk_ids, 64, e)
    sid, eid, npp = gu.dev_i32(sorted_ids), gu.dev_i32(expert_ids), gu.dev_i32(np.array([int(past[0])], dtype=np.int32))
    c = torch.zeros((tokens * top_k, n), dtype=torch.bfloat16, device=DEV)
    workspace = torch.zeros(1024, dtype=torch.int32, device=DEV)
    nbytes = lib.sonar_moe_marlin_gemm_scratch_bytes(sid.numel(), 64, n, k)
    scratch = torch.empty(max(nbytes, 16), dtype=torch.uint8, device=DEV)
    _lib.check(lib.sonar_moe_wna16_marlin_gemm(
        gu.ptr(a), gu.ptr(c), gu.ptr(native), _lib.LAYOUT_GFX950, None, gu.ptr(scales), None, None, None, gu.ptr(workspace),
        workspace.numel(), gu.ptr(scratch), nbytes, gu.ptr(sid), sid.numel(), gu.ptr(eid), gu.ptr(npp), None, 64, top_k, 0, e,
        _lib.DTYPE_BF16, b_type, tokens, n, k, 1, 1, 0, 1, gu.stream()))
    for expert in range(e):
        slots = np.nonzero(topk_ids.reshape(-1) == expert)[0][:16]
        rows = a[torch.from_numpy(slots // top_k).to(DEV)].contiguous()
        dense = torch.empty((len(slots), n), dtype=torch.bfloat16, device=DEV)
        room = torch.empty(max(lib.sonar_marlin_gemm_scratch_bytes(len(slots), n, k), 16), dtype=torch.uint8, device=DEV)
        _lib.check(lib.sonar_marlin_gemm(
            gu.ptr(rows), k, gu.ptr(dense), gu.ptr(native[expert]), _lib.LAYOUT_GFX950, None, gu.ptr(scales[expert]), None, None,
            None, gu.ptr(workspace), workspace.numel(), gu.ptr(room), room.numel(), _lib.DTYPE_BF16, b_type, len(slots), n, k, 1, 1,
            0, 1, gu.stream()))
        got, want = c[torch.from_numpy(slots).to(DEV)].double(), dense.double()
        # numbers of eight bits are 2^-7 of their power of two apart, and the rounding error is evenly spread
        rounding = (torch.exp2(torch.floor(torch.log2(want.abs().clamp_min(1e-30)))) * 2.0 ** -7 / 12.0 ** 0.5).norm()
        assert (got - want).norm() <= 0.35 * rounding, (expert, float((got - want).norm() / rounding))


if __name__ == "__main__":
    for shape in SHAPES:
        for is_fp8 in (False, True):
            print(*shape, is_fp8, flush=True)
            _check(*shape, is_fp8)
    print("all shapes ok", flush=True)
