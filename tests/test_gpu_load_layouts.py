"""The layout kernels of weight loading against the torch expressions they replace (which serve CPU
tensors and are checked against the oracle in test_host_logic.py) and against the oracle."""
from __future__ import annotations

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from oracle import marlin_oracle as mo

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _words(rng, *shape):
    return torch.from_numpy(rng.integers(-2 ** 31, 2 ** 31, size=shape, dtype=np.int64).astype(np.int32))


# tile counts that are no multiple of a workgroup's, one tile in all, experts whose tiles share a workgroup
@pytest.mark.parametrize("experts,k,n", [(1, 16, 64), (3, 48, 192), (5, 128, 320), (2, 256, 1024)])
@pytest.mark.parametrize("kind", ["gptq", "act_order", "awq"])
def test_stacked_repack_is_the_repack_of_every_matrix(kind, experts, k, n):
    from sonar_amd import ops
    rng = np.random.default_rng(experts * k + n)
    perm = np.stack([rng.permutation(k) for _ in range(experts)]).astype(np.int32)
    if kind == "awq":
        w = _words(rng, experts, k, n // 8)
        got = ops.awq_marlin_moe_repack(w.to(DEV), torch.empty((experts, 0), dtype=torch.int32, device=DEV), k, n, 4)
        want = [mo.awq_marlin_repack(w[e].numpy(), k, n) for e in range(experts)]
    else:
        w = _words(rng, experts, k // 8, n)
        p = perm if kind == "act_order" else np.empty((experts, 0), np.int32)
        got = ops.gptq_marlin_moe_repack(w.to(DEV), torch.from_numpy(p).to(DEV), k, n, 4)
        want = [mo.gptq_marlin_repack(w[e].numpy(), perm[e] if kind == "act_order" else None, k, n) for e in range(experts)]
    assert np.array_equal(got.cpu().numpy(), np.stack(want))


# buffers that are aligned as words and no better: views that begin inside a larger tensor
@pytest.mark.parametrize("offset", [1, 2, 3])
def test_repack_of_views_that_begin_at_any_word(offset):
    from sonar_amd import _lib, ops
    from tests import gpu_util as gu
    e, k, n = 2, 48, 192
    rng = np.random.default_rng(offset)
    words = e * k * n // 8
    flat = _words(rng, words + 8).to(DEV)
    perm = np.stack([rng.permutation(k) for _ in range(e)]).astype(np.int32)
    none = torch.empty((e, 0), dtype=torch.int32, device=DEV)
    gptq, awq = flat[offset:offset + words].view(e, k // 8, n), flat[offset:offset + words].view(e, k, n // 8)
    assert gptq.data_ptr() % 16 == 4 * offset
    host_gptq, host_awq = gptq.cpu().numpy(), awq.cpu().numpy()
    for p, got in ((None, ops.gptq_marlin_moe_repack(gptq, none, k, n, 4)),
                   (perm, ops.gptq_marlin_moe_repack(gptq, torch.from_numpy(perm).to(DEV), k, n, 4))):
        want = np.stack([mo.gptq_marlin_repack(host_gptq[i], None if p is None else p[i], k, n) for i in range(e)])
        assert np.array_equal(got.cpu().numpy(), want)
    want = np.stack([mo.awq_marlin_repack(host_awq[i], k, n) for i in range(e)])
    assert np.array_equal(ops.awq_marlin_moe_repack(awq, none, k, n, 4).cpu().numpy(), want)
    codes, _ = torch.ops.sonar_amd.awq_to_standard(awq[0], awq[1][:2].contiguous())
    assert np.array_equal(ops.gptq_marlin_repack(codes, none[0], k, n, 4).cpu().numpy(), want[0])
    lib = _lib.load()
    out = torch.empty(words + 4, dtype=torch.int32, device=DEV)[offset:offset + words]
    _lib.check(lib.sonar_awq_marlin_moe_repack(gu.ptr(awq), gu.ptr(out), e, k, n, gu.stream()))
    assert np.array_equal(out.cpu().numpy(), want.reshape(-1))
    _lib.check(lib.sonar_awq_to_gptq(gu.ptr(awq), gu.ptr(out), k, n, gu.stream()))
    assert torch.equal(out[:words // e], codes.reshape(-1))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,n,group", [(1, 64, -1), (3, 192, 128), (33, 1088, 64), (256, 4096, 32)])
def test_permute_scales_and_bias(dtype, rows, n, group):
    from sonar_amd import marlin_utils as mu
    s = torch.randn(rows, n).to(dtype)
    k = 100000
    assert torch.equal(mu.marlin_permute_scales(s.to(DEV), k, n, group).cpu(), mu.marlin_permute_scales(s, k, n, group))
    assert torch.equal(mu.marlin_permute_scales(s.t().contiguous().to(DEV).t(), k, n, group).cpu(),
                       mu.marlin_permute_scales(s, k, n, group))
    assert torch.equal(mu.marlin_permute_bias(s[0].to(DEV)).cpu(), mu.marlin_permute_bias(s[0]))
    e = torch.stack([s, -s])
    assert torch.equal(mu.marlin_moe_permute_scales(e.to(DEV), k, n, group).cpu(), mu.marlin_moe_permute_scales(e, k, n, group))


@pytest.mark.parametrize("groups,n", [(1, 64), (7, 192), (32, 1024)])
@pytest.mark.parametrize("a8", [False, True])
def test_zero_points(groups, n, a8):
    from sonar_amd import marlin_utils as mu
    z = _words(np.random.default_rng(groups + n), 3, groups, n // 8)
    for fn in (mu.moe_awq_to_marlin_zero_points, mu.moe_packed_to_marlin_zero_points):
        assert torch.equal(fn(z.to(DEV), groups, n, 4, a8).cpu(), fn(z, groups, n, 4, a8))
    assert torch.equal(mu.awq_to_marlin_zero_points(z[0].to(DEV), groups, n, 4, a8).cpu(),
                       mu.awq_to_marlin_zero_points(z[0], groups, n, 4, a8))


@pytest.mark.parametrize("k,n,group", [(128, 64, 128), (256, 320, 64), (1024, 1088, 32), (128, 128, 8)])
def test_awq_checkpoint_is_loaded_as_on_the_cpu(k, n, group):
    from sonar_amd import marlin_linear as ml
    from sonar_amd import ops
    from sonar_amd.scalar_type import scalar_types
    rng = np.random.default_rng(k + n)
    qw, qz = _words(rng, k, n // 8), _words(rng, k // group, n // 8)
    cpu, gpu = (SimpleNamespace(qweight=qw.to(d), qzeros=qz.to(d)) for d in ("cpu", DEV))
    ml.convert_awq_to_standard_format(cpu)
    ml.convert_awq_to_standard_format(gpu)
    assert torch.equal(gpu.qweight.cpu(), cpu.qweight) and torch.equal(gpu.qzeros.cpu(), cpu.qzeros)
    if group < 32:
        return
    gpu.scales = torch.rand(k // group, n, device=DEV).to(torch.float16)
    cfg = ml.MPLinearLayerConfig((k, n), (k, n), scalar_types.uint4, torch.float16, group, True, False)
    ml.MarlinLinearKernel(cfg).process_weights_after_loading(gpu)
    z = mo.awq_to_marlin_zero_points(qz.numpy(), k // group, n)
    assert np.array_equal(gpu.qzeros.cpu().numpy(), z)
    assert torch.equal(gpu.qweight, ops.awq_marlin_repack(qw.to(DEV), k, n, 4))


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="two GPUs")
def test_awq_tensors_on_two_gpus():
    """Codes and zero points are converted where they lie: one launch takes both only where they lie together."""
    from sonar_amd import marlin_linear as ml
    qw, qz = _words(np.random.default_rng(1), 256, 40), _words(np.random.default_rng(2), 4, 40)
    cpu = SimpleNamespace(qweight=qw, qzeros=qz)
    gpu = SimpleNamespace(qweight=qw.to("cuda:0"), qzeros=qz.to("cuda:1"))
    ml.convert_awq_to_standard_format(cpu)
    ml.convert_awq_to_standard_format(gpu)
    assert gpu.qweight.device.index == 0 and gpu.qzeros.device.index == 1
    assert torch.equal(gpu.qweight.cpu(), cpu.qweight) and torch.equal(gpu.qzeros.cpu(), cpu.qzeros)
