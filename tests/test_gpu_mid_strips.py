"""The four-strip workgroups of marlin_mid_gemm, each case with the strips that it ran in: grouped calls of every block size whose last
workgroup has one to four strips of its own, at the fewest rows of K that the form is given and at an odd number of units; the dense
shapes of test_gpu_mid_four_strips; and the gated activation where the ranges meet, in layers whose gate and up rows are in that
kernel and are not written."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import marlin_oracle as mo
from sonar_amd import _lib, fused_moe, marlin_utils as mu, ops
from sonar_amd.scalar_type import scalar_types
from tests import gpu_util as gu
from tests import test_gpu_mid_four_strips as dense
from tests import test_gpu_moe as tm
from tests.test_gpu_moe_routed import _experts

pytestmark = pytest.mark.gpu


def _ran_in(strips: int, grouped: bool = True) -> None:
    lib = _lib.load()
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:   # (rounds of workgroups on 256 compute units)
        assert not grouped or lib.sonar_marlin_last_grouped_kernel() == _lib.GROUPED_MID
        assert lib.sonar_marlin_last_mid_strips() == strips


@pytest.mark.parametrize("m,slots", [(200, 32), (296, 48), (400, 64)])
@pytest.mark.parametrize("k,n", [(512, 2240), (512, 2304), (512, 2368), (512, 2432), (1664, 2368)])   # 35 to 38 strips
@pytest.mark.parametrize("dtype,zp,group", [("fp16", False, 128), ("bf16", True, -1)])
def test_four_strips(m, slots, k, n, dtype, zp, group):
    tm.test_moe_gemm_within_tolerance((m, 16, 2, k, n, group, dtype, zp, False, zp, slots, not zp))
    _ran_in(4)


# ... and the types and groups that those leave out
@pytest.mark.parametrize("m,slots", [(200, 32), (296, 48), (400, 64)])
@pytest.mark.parametrize("dtype,zp,group", [("fp16", False, -1), ("fp16", True, 128), ("fp16", True, -1), ("bf16", False, 128), ("bf16", False, -1),
                                            ("bf16", True, 128)])
def test_four_strips_in_every_form(m, slots, dtype, zp, group):
    tm.test_moe_gemm_within_tolerance((m, 16, 2, 640, 2368, group, dtype, zp, False, zp, slots, not zp))
    _ran_in(4)


# fewer than a round of two strips a workgroup, and K below 512
@pytest.mark.parametrize("m,e,k,n,slots", [(400, 16, 512, 2048, 64), (296, 16, 384, 2432, 48)])
def test_two_strips(m, e, k, n, slots):
    tm.test_moe_gemm_within_tolerance((m, e, 2, k, n, 128, "bf16", False, False, False, slots, True))
    _ran_in(2)


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("zp", [False, True])
@pytest.mark.parametrize("m,k,n,group", [(65, 640, 24640, 128), (128, 1408, 24768, -1), (97, 1152, 16576, 128)])
def test_dense(m, k, n, group, zp, dtype):
    dense.test_against_the_oracle(m, k, n, group, zp, dtype)
    _ran_in(4, grouped=False)


# blocks of 32, 48 and 64 slots; halves of an odd number of strips
@pytest.mark.parametrize("kind,group,dtype", [("uint4b8", 128, torch.float16), ("uint4", 128, torch.bfloat16), ("mxfp4", 32, torch.bfloat16)])
@pytest.mark.parametrize("tokens,k,inter,strips", [(200, 512, 832, 2), (296, 512, 576, 2), (400, 512, 576, 2), (400, 640, 960, 2),
                                                   (296, 640, 1344, 4), (400, 1152, 1600, 4)])
def test_gated_activation(tokens, k, inter, strips, kind, group, dtype):
    e, rows = 16, 2 * tokens
    gen = torch.Generator(device=gu.DEV).manual_seed(tokens + k)
    w1, s1, z1 = _experts(gen, kind, e, k, 2 * inter, group, dtype)
    w2, s2, z2 = _experts(gen, kind, e, inter, k, min(group, 64), dtype)
    bias1 = (torch.randn((e, 2 * inter), device=gu.DEV, generator=gen) * 0.1).to(dtype)
    x = torch.randn((tokens, k), device=gu.DEV, generator=gen).to(dtype) * 0.1
    weights, ids = torch.topk(torch.softmax(torch.randn((tokens, e), device=gu.DEV, generator=gen), dim=1), 2, dim=1)
    wtype = {"uint4b8": scalar_types.uint4b8, "uint4": scalar_types.uint4, "mxfp4": scalar_types.float4_e2m1f}[kind]
    assert 2 * inter > k
    for activation, on_input in (("swigluoai", False), ("silu", False), ("silu", True)):
        def layer(**kw):
            return fused_moe.fused_marlin_moe(x, w1, w2, bias1, None, s1, s2, weights.contiguous(), ids.to(torch.int32), wtype.id, on_input,
                                              activation=activation, w1_zeros=z1, w2_zeros=z2, **kw)
        between = torch.empty((rows, inter), dtype=dtype, device=gu.DEV)

        def after(name, out, rows_in, **kw):   # behind the GEMM of the gate and up rows
            _ran_in(strips)
            fused_moe.apply_moe_activation(name, out, rows_in, **kw)
            between.copy_(out)

        cache13 = torch.full((rows * 2 * inter,), -7.0, dtype=dtype, device=gu.DEV)
        cache2 = torch.empty((rows * inter,), dtype=dtype, device=gu.DEV)
        got = layer(intermediate_cache13=cache13, intermediate_cache2=cache2)
        assert bool((cache13[rows * k:] == -7.0).all()), activation   # the gate and up rows were not written
        want = layer(activation_func=after)
        assert bool(torch.isfinite(want).all())
        assert torch.equal(cache2.view(rows, inter), between) and torch.equal(got, want), activation


# a round or more of blocks of 32 slots: the decode kernel's where it forms the activation, and only there
@pytest.mark.parametrize("n,activation,limit,written,kernel", [
    (2304, "SILU", 0.0, 1, "DECODE"), (2304, "SWIGLUOAI", 7.0, 1, "DECODE"), (2368, "SWIGLUOAI", 7.0, 1, "DECODE"),
    (2304, "GELU", 0.0, 0, "MID"), (2368, "SILU", 0.0, 0, "MID"), (2304, "SWIGLUOAI", 0.0, 0, "MID")])
def test_an_activation_that_no_kernel_forms_changes_no_route(n, activation, limit, written, kernel):
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("rounds of workgroups on 256 compute units")
    kinds = {"SILU": 0, "GELU": 2, "SWIGLUOAI": 4}
    m, e, top_k, k, slots = 200, 16, 2, 512, 32
    lib = _lib.load()
    ex = tm.Experts(5, e, k, n, 128, "bf16")
    sorted_ids, expert_ids, past = mo.moe_align_block_size(tm.route(3, m, e, top_k)[0], slots, e)
    sid, eid, npp = (gu.dev_i32(np.asarray(x).reshape(-1)) for x in (sorted_ids, expert_ids, past))
    a = gu.dev_bits16(mo.make_activations(4, m, k, "bf16"), "bf16")

    def call(out, answer):
        c = torch.full((m * top_k, n), -7.0, dtype=torch.bfloat16, device=gu.DEV)
        _lib.check(lib.sonar_moe_wna16_marlin_gemm_gated(
            gu.ptr(a), gu.ptr(c), gu.ptr(ex.native), _lib.LAYOUT_GFX950, None, gu.ptr(ex.scales), None, None, None, None, None, 0,
            gu.ptr(sid), sid.numel(), gu.ptr(eid), gu.ptr(npp), None, slots, top_k, 0, e, _lib.DTYPE_BF16, ex.b_type, m, n, k, ex.groups, 1,
            gu.ptr(out), kinds[activation], limit, 1.702, answer, None, None, gu.stream()))
        torch.cuda.synchronize()
        return c, lib.sonar_marlin_last_grouped_kernel()

    done = ctypes.c_int(5)
    plain, ran = call(None, ctypes.byref(done))
    assert ran == _lib.GROUPED_MID and done.value == 0
    out = torch.full((m * top_k, n // 2), -7.0, dtype=torch.bfloat16, device=gu.DEV)
    c, ran = call(out, ctypes.byref(done))
    assert done.value == written and ran == getattr(_lib, "GROUPED_" + kernel)
    assert torch.equal(c, torch.full_like(c, -7.0) if written else plain) and bool((out == -7.0).all()) != bool(written)


# up to 64 rows of a matrix of more than 256 pairs of strips: one round of four strips, the longer the fuller it is and not the more bytes the
# matrix has; the widest of these were left to kernels that take 1.1 to 1.4 times as long.  Against the decode kernel, 16 rows at a time.
@pytest.mark.parametrize("m,k,n,dtype", [(49, 7424, 51968, torch.float16), (62, 2944, 46592, torch.bfloat16), (64, 8192, 57344, torch.bfloat16)])
def test_wide_matrices(m, k, n, dtype):
    gen = torch.Generator(device=gu.DEV).manual_seed(m)
    q = torch.randint(-2 ** 31, 2 ** 31 - 1, (k // 16, 2 * n), dtype=torch.int32, device=gu.DEV, generator=gen)
    s = (torch.rand((k // 128, n), device=gu.DEV, generator=gen) * 9e-3 + 1e-3).to(dtype)
    a = torch.randn((m, k), device=gu.DEV, generator=gen).to(dtype)
    empty = torch.empty(0, dtype=torch.int32, device=gu.DEV)
    workspace = mu.marlin_make_workspace_new(torch.device(gu.DEV))

    def gemm(rows):
        return ops.marlin_gemm(rows, None, q, None, s, None, None, empty, empty, empty, workspace, scalar_types.uint4b8, rows.shape[0], n, k,
                               True, False, True, False)
    got = gemm(a)
    _ran_in(4, grouped=False)
    want = torch.cat([gemm(a[i:i + 16]) for i in range(0, m, 16)])
    assert _lib.load().sonar_marlin_last_mid_strips() == 0
    scale = float(want.float().abs().max())
    assert bool(torch.isfinite(want).all()) and float((got.float() - want.float()).abs().max()) <= 1e-2 * scale
