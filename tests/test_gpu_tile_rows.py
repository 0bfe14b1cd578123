"""Rows of results of the wide tile kernel leave through LDS as 16-byte pieces: a matrix C that is aligned to 8 bytes only
gets the bits of an aligned one, dense (ragged last tiles of rows and columns, both tile sizes) and grouped (rows scattered by
the routing), and nothing around it."""
from __future__ import annotations

import pytest
import torch

from sonar_amd import marlin_utils as mu
from sonar_amd import ops
from sonar_amd.scalar_type import scalar_types

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _c_views(m, n, dtype, guard=64):
    for offset in (0, 4):   # the ops ask for 8 bytes
        whole = torch.full((m * n + 2 * guard,), -7.0, dtype=dtype, device=DEV)
        yield whole, whole[guard + offset:guard + offset + m * n].view(m, n), guard + offset


def _untouched(whole, first, count):
    return bool((whole[:first] == -7.0).all()) and bool((whole[first + count:] == -7.0).all())


def _weights(gen, experts, k, n, dtype):
    q = torch.randint(-2 ** 31, 2 ** 31 - 1, (experts, k // 16, 2 * n), dtype=torch.int32, device=DEV, generator=gen)
    s = (torch.rand((experts, k // 128, n), device=DEV, generator=gen) * 9e-3 + 1e-3).to(dtype)
    return q, s


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,k,n", [(1025, 4096, 4160), (2817, 128, 8192), (300, 14336, 1088)])
def test_dense(dtype, m, k, n):
    gen = torch.Generator(device=DEV).manual_seed(m)
    q, s = _weights(gen, 1, k, n, dtype)
    a = torch.randn((m, k), device=DEV, generator=gen).to(dtype)
    empty = torch.empty(0, dtype=torch.int32, device=DEV)
    ws = mu.marlin_make_workspace_new(torch.device(DEV))
    want = None
    for whole, c, first in _c_views(m, n, dtype):
        out = ops.marlin_gemm(a, c, q[0], None, s[0], None, None, empty, empty, empty, ws, scalar_types.uint4b8, m, n, k,
                              True, False, True, False)
        assert out.data_ptr() == c.data_ptr()
        want = c.clone() if want is None else want
        assert torch.equal(c, want) and bool(torch.isfinite(want).all()) and _untouched(whole, first, m * n)


@pytest.mark.parametrize("mul_topk", [False, True])
def test_grouped(mul_topk):
    from sonar_amd import fused_moe
    m, k, n, e, top_k, dtype = 1100, 192, 1088, 3, 2, torch.bfloat16
    gen = torch.Generator(device=DEV).manual_seed(5)
    q = torch.randint(-2 ** 31, 2 ** 31 - 1, (e, k // 16, 2 * n), dtype=torch.int32, device=DEV, generator=gen)
    s = (torch.rand((e, k // 64, n), device=DEV, generator=gen) * 9e-3 + 1e-3).to(dtype)
    a = torch.randn((m, k), device=DEV, generator=gen).to(dtype)
    weights, ids = torch.topk(torch.softmax(torch.randn((m, e), device=DEV, generator=gen), dim=1), top_k, dim=1)
    sorted_ids, expert_ids, past = fused_moe.moe_align_block_size(ids.to(torch.int32), 64, e)
    ws = mu.marlin_make_workspace_new(torch.device(DEV), 4)
    want = None
    for whole, c, first in _c_views(m * top_k, n, dtype):
        ops.moe_wna16_marlin_gemm(a, c, q, None, s, None, None, None, None, None, ws, sorted_ids, expert_ids, past,
                                  weights.contiguous(), moe_block_size=64, top_k=top_k, mul_topk_weights=mul_topk,
                                  b_q_type=scalar_types.uint4b8, size_m=m, size_n=n, size_k=k, is_k_full=True,
                                  use_atomic_add=False, use_fp32_reduce=True, is_zp_float=False)
        want = c.clone() if want is None else want
        assert torch.equal(c, want) and bool((want != -7.0).all()) and _untouched(whole, first, m * top_k * n)


def test_rows_of_a_too_far_apart_for_32_bit_offsets():
    """Rows 64 MiB apart: the kernels that take such calls, against the same rows side by side (two roundings to fp16 differ)."""
    m, k, n, dtype = 150, 8192, 1088, torch.float16
    gen = torch.Generator(device=DEV).manual_seed(1)
    q, s = _weights(gen, 1, k, n, dtype)
    far = torch.empty_strided((m, k), (1 << 25, 1), dtype=dtype, device=DEV)
    far.copy_(torch.randn((m, k), device=DEV, generator=gen))
    empty = torch.empty(0, dtype=torch.int32, device=DEV)
    ws = mu.marlin_make_workspace_new(torch.device(DEV))
    got, want = (ops.marlin_gemm(a, None, q[0], None, s[0], None, None, empty, empty, empty, ws, scalar_types.uint4b8, m, n, k,
                                 True, False, True, False).double() for a in (far, far.contiguous()))
    assert float((got - want).norm() / want.norm()) < 2e-3


# the row strides up to which the wide tile kernel's 32-bit offsets reach, and the first beyond: both tile sizes, ragged rows
@pytest.mark.parametrize("wtype", ["uint4b8", "uint8b128", "float8_e4m3fn"])
@pytest.mark.parametrize("m,k,n", [(200, 512, 32832), (400, 256, 8256)])
def test_strides_of_rows_of_a(wtype, m, k, n):
    dtype = torch.float16
    gen = torch.Generator(device=DEV).manual_seed(m)
    words = 2 if wtype == "uint4b8" else 4
    q = torch.randint(-2 ** 31, 2 ** 31 - 1, (k // 16, words * n), dtype=torch.int32, device=DEV, generator=gen) & 0x77777777
    s = (torch.rand((k // 128, n), device=DEV, generator=gen) * (1e-3 if words == 4 else 9e-3) + 1e-4).to(dtype)
    near = torch.randn((m, k), device=DEV, generator=gen).to(dtype)
    empty = torch.empty(0, dtype=torch.int32, device=DEV)
    ws = mu.marlin_make_workspace_new(torch.device(DEV))

    def call(a):
        return ops.marlin_gemm(a, None, q, None, s, None, None, empty, empty, empty, ws, getattr(scalar_types, wtype), m, n, k,
                               True, False, True, False)

    want = call(near)
    assert bool(torch.isfinite(want).all())
    for stride in (1 << 23, (1 << 25) - 8, 1 << 25):
        far = torch.empty_strided((m, k), (stride, 1), dtype=dtype, device=DEV)
        got = call(far.copy_(near))
        del far
        if stride < 1 << 25:
            assert torch.equal(got, want), stride
        else:   # another kernel: two roundings to fp16 differ
            assert float((got.double() - want.double()).norm() / want.double().norm()) < 2e-3
