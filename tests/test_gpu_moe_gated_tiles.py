"""The grouped tile kernels form the gated activation of their rows themselves: a layer gives the bits of the GEMM and the
activation kernel after one another, in every weight format and kind of launch (both tile sizes; one, for NVFP4 and 8-bit codes with
groups of 32 rows), with a ragged last tile of columns (alternating gate
and up only: halves need whole tiles), experts without rows, a bias and the routing weight on the input; the gate and up rows are
not written then.  The row tiles of both GEMMs of a layer come from one launch, whichever of them may cut its tiles along K.
Activations and widths that the tiles do not take go the old way."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import marlin_oracle as mo
from sonar_amd import _lib, fused_moe
from sonar_amd.scalar_type import scalar_types
from tests import gpu_util as gu
from tests import test_gpu_moe as tm

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _experts(gen, kind, e, k, n, dtype):
    """Random experts in the Marlin layout: weights, scales, zero points."""
    words = 2 if kind in ("uint4b8", "uint4", "mxfp4", "nvfp4") else 4
    q = torch.randint(-2 ** 31, 2 ** 31 - 1, (e, k // 16, words * n), dtype=torch.int32, device=DEV, generator=gen)
    if kind == "mxfp4":
        s = torch.randint(117, 122, (e, k // 32, n), dtype=torch.uint8, device=DEV, generator=gen).view(torch.float8_e8m0fnu)
    elif kind == "nvfp4":   # as the loading leaves them: the upper bytes of 1 to 4 times 2^7 in fp16, shifted by one
        s = torch.randint(0xB0, 0xC0, (e, k // 16, n), dtype=torch.uint8, device=DEV, generator=gen).view(torch.float8_e4m3fn)
    elif kind == "fp8":     # a scale a column, the codes' exponent bias in it; no code that is NaN
        q &= 0x77777777
        s = (torch.rand((e, 1, n), device=DEV, generator=gen) * 2.56e-2 + 2.56e-3).to(dtype)
    elif kind == "uint8b128g32":
        s = ((torch.rand((e, k // 32, n), device=DEV, generator=gen) * 9e-3 + 1e-3) / 16).to(dtype)
    else:
        s = (torch.rand((e, k // 64, n), device=DEV, generator=gen) * 9e-3 + 1e-3).to(dtype)
        s = s / 16 if kind == "uint8b128" else s
    z = None
    if kind == "uint4":
        z = torch.randint(-2 ** 31, 2 ** 31 - 1, (e, k // 64, n // 8), dtype=torch.int32, device=DEV, generator=gen)
    return q, s, z


@pytest.mark.parametrize("kind,dtype", [("uint4b8", torch.float16), ("uint4", torch.bfloat16), ("mxfp4", torch.bfloat16),
                                        ("uint8b128", torch.float16)])
@pytest.mark.parametrize("activation,inter,k,in_tiles", [("silu", 384, 320, True), ("silu", 320, 320, False),
                                                         ("swigluoai", 384, 192, True), ("swigluoai", 352, 320, True),
                                                         ("gelu", 384, 320, False), ("silu", 1024, 1024, True), ("swigluoai", 576, 1024, True),
                                                         ("silu", 1024, 320, True), ("gelu", 1024, 1024, False)])
@pytest.mark.parametrize("on_input", [False, True])
def test_layer(kind, dtype, activation, inter, k, in_tiles, on_input):
    _check_layer(kind, dtype, activation, inter, k, in_tiles, on_input)


@pytest.mark.parametrize("kind,dtype", [("nvfp4", torch.float16), ("nvfp4", torch.bfloat16), ("uint8b128g32", torch.bfloat16),
                                        ("fp8", torch.float16)])
@pytest.mark.parametrize("activation,inter,k,in_tiles", [("silu", 384, 320, True), ("swigluoai", 384, 192, True),
                                                         ("swigluoai", 576, 1024, True), ("silu", 320, 320, False)])
def test_layer_of_other_formats(kind, dtype, activation, inter, k, in_tiles):
    _check_layer(kind, dtype, activation, inter, k, in_tiles, inter == 384)


def _check_layer(kind, dtype, activation, inter, k, in_tiles, on_input):
    if kind != "mxfp4" and inter % 64:   # the down projection's groups
        inter = 448
    m, e, top_k = 1500 if kind == "mxfp4" else 700, 6, 2   # (MXFP4: more than marlin_mid_gemm takes)
    gen = torch.Generator(device=DEV).manual_seed(inter + k)
    w1, s1, z1 = _experts(gen, kind, e, k, 2 * inter, dtype)
    w2, s2, z2 = _experts(gen, kind, e, inter, k, dtype)
    bias1 = (torch.randn((e, 2 * inter), device=DEV, generator=gen) * 0.1).to(dtype)
    x = torch.randn((m, k), device=DEV, generator=gen).to(dtype)
    logits = torch.randn((m, e), device=DEV, generator=gen)
    logits[:, 0] += 3.0    # most tokens: tiles of 256 rows
    logits[:, 2] -= 100.0  # none
    weights, ids = torch.topk(torch.softmax(logits, dim=1), top_k, dim=1)
    weights, ids = weights.contiguous(), ids.to(torch.int32)
    wtype = {"uint4b8": scalar_types.uint4b8, "uint4": scalar_types.uint4, "mxfp4": scalar_types.float4_e2m1f,
             "uint8b128": scalar_types.uint8b128, "uint8b128g32": scalar_types.uint8b128, "fp8": scalar_types.float8_e4m3fn,
             "nvfp4": scalar_types.float4_e2m1f}[kind]
    global_scale = None
    if kind == "nvfp4":
        global_scale = torch.rand(e, device=DEV, generator=gen) * 1e-3 + 1e-3
        global_scale *= 2.0 ** (7 if dtype == torch.float16 else 119)
    assert fused_moe.moe_block_size(m, top_k, e) == 64 and 2 * inter > k or k == 1024

    def layer(**kw):
        return fused_moe.fused_marlin_moe(x, w1, w2, bias1, None, s1, s2, weights, ids, wtype.id, on_input,
                                          activation=activation, w1_zeros=z1, w2_zeros=z2, global_scale1=global_scale,
                                          global_scale2=global_scale, **kw)

    rows = m * top_k
    cache13 = torch.full((rows * max(2 * inter, k),), -7.0, dtype=dtype, device=DEV)
    cache2 = torch.empty((rows * inter,), dtype=dtype, device=DEV)
    got = layer(intermediate_cache13=cache13, intermediate_cache2=cache2)
    if 2 * inter > k:
        assert bool((cache13[rows * k:] == -7.0).all()) == in_tiles
    between = torch.empty((rows, inter), dtype=dtype, device=DEV)

    def after(name, out, rows_in, **kw):   # a function of the caller's own: two calls, the GEMM and the activation
        fused_moe.apply_moe_activation(name, out, rows_in, **kw)
        between.copy_(out)

    want = layer(activation_func=after)
    assert bool(torch.isfinite(want.float()).all())
    assert torch.equal(cache2.view(rows, inter), between)
    assert torch.equal(got, want)


def test_many_blocks():
    """More blocks of slots than the smaller form of the table kernel has threads."""
    m, e, top_k, k, inter, dtype = 9001, 5, 2, 320, 1024, torch.bfloat16
    gen = torch.Generator(device=DEV).manual_seed(2)
    w1, s1, _ = _experts(gen, "uint4b8", e, k, 2 * inter, dtype)
    w2, s2, _ = _experts(gen, "uint4b8", e, inter, k, dtype)
    x = torch.randn((m, k), device=DEV, generator=gen).to(dtype)
    weights, ids = torch.topk(torch.rand((m, e), device=DEV, generator=gen), top_k, dim=1)
    args = (x, w1, w2, None, None, s1, s2, weights.contiguous(), ids.to(torch.int32), scalar_types.uint4b8.id)
    assert torch.equal(fused_moe.fused_marlin_moe(*args),
                       fused_moe.fused_marlin_moe(*args, activation_func=fused_moe.apply_moe_activation))


def test_input_in_the_place_of_the_rows_between():
    """hidden_states inside intermediate_cache2: the GEMM reads all of it before anything is written there."""
    m, e, top_k, k, inter, dtype = 700, 3, 2, 320, 384, torch.bfloat16
    gen = torch.Generator(device=DEV).manual_seed(1)
    w1, s1, _ = _experts(gen, "uint4b8", e, k, 2 * inter, dtype)
    w2, s2, _ = _experts(gen, "uint4b8", e, inter, k, dtype)
    cache2 = torch.empty((m * top_k * inter,), dtype=dtype, device=DEV)
    x = torch.randn((m, k), device=DEV, generator=gen).to(dtype)
    inside = cache2[:m * k].view(m, k)
    weights, ids = torch.topk(torch.rand((m, e), device=DEV, generator=gen), top_k, dim=1)
    weights, ids = weights.contiguous(), ids.to(torch.int32)
    want = fused_moe.fused_marlin_moe(x, w1, w2, None, None, s1, s2, weights, ids, scalar_types.uint4b8.id)
    inside.copy_(x)
    got = fused_moe.fused_marlin_moe(inside, w1, w2, None, None, s1, s2, weights, ids, scalar_types.uint4b8.id,
                                     intermediate_cache2=cache2)
    assert torch.equal(got, want)


class _Tables(ctypes.Structure):
    _fields_ = [("table", ctypes.c_void_p), ("table_bytes", ctypes.c_size_t), ("size_n", ctypes.c_int64), ("size_k", ctypes.c_int64),
                ("num_groups", ctypes.c_int64), ("built", ctypes.c_int), ("tiles_n", ctypes.c_int), ("k_steps", ctypes.c_int),
                ("may_split", ctypes.c_int), ("expert_ids", ctypes.c_void_p), ("sorted_len", ctypes.c_int64)]


def test_row_tiles_laid_down_by_another_call_are_used_once():
    """A second call with the same struct, the routing changed in place meanwhile, has to build its own."""
    lib = _lib.load()
    m, e, top_k, k, n, bs = 1400, 4, 1, 256, 320, 64
    ex = tm.Experts(7, e, k, n, 64, "bf16")
    a = torch.randn((m, k), device=DEV, generator=torch.Generator(device=DEV).manual_seed(4)).to(torch.bfloat16)
    routes = []
    for seed in (1, 2):   # the second: most slots of the last expert
        ids = tm.route(seed, m, e, top_k)[0]
        if seed == 2:
            ids[:1000] = e - 1
        routes.append(mo.moe_align_block_size(ids, bs, e))
    sid, eid, npp = (gu.dev_i32(np.asarray(x).reshape(-1)) for x in routes[0])
    tables = _Tables(size_n=n, size_k=k, num_groups=ex.groups)
    room = torch.empty(lib.sonar_moe_marlin_gemm_scratch_bytes(sid.numel(), bs, n, 64), dtype=torch.uint8, device=DEV)
    tables.table, tables.table_bytes = room.data_ptr(), room.numel()

    def call(next_call=None, ready=None):
        c = torch.zeros((m, n), dtype=torch.bfloat16, device=DEV)
        scratch = torch.empty(lib.sonar_moe_marlin_gemm_scratch_bytes(sid.numel(), bs, n, k), dtype=torch.uint8, device=DEV)
        written = ctypes.c_int(-1)
        _lib.check(lib.sonar_moe_wna16_marlin_gemm_gated(
            gu.ptr(a), gu.ptr(c), gu.ptr(ex.native), _lib.LAYOUT_GFX950, None, gu.ptr(ex.scales), None, None, None, None, gu.ptr(scratch),
            scratch.numel(), gu.ptr(sid), sid.numel(), gu.ptr(eid), gu.ptr(npp), None, bs, top_k, 0, e, _lib.DTYPE_BF16, ex.b_type, m,
            n, k, ex.groups, 1, None, 0, 0.0, 0.0, ctypes.byref(written), next_call, ready, gu.stream()))
        torch.cuda.synchronize()
        assert written.value == 0 and lib.sonar_marlin_last_grouped_kernel() == _lib.GROUPED_TILE
        return c

    want = call()
    assert torch.equal(call(next_call=ctypes.byref(tables)), want) and tables.built == 1
    assert torch.equal(call(ready=ctypes.byref(tables)), want) and tables.built == 0
    for t, x in zip((sid, eid, npp), routes[1]):
        t.copy_(gu.dev_i32(np.asarray(x).reshape(-1)))
    assert torch.equal(call(ready=ctypes.byref(tables)), call())
