"""AWQ checkpoints with as many groups as words of zero points in a row (K / group == N / 8), where the shape of the converted
zero points does not say that they are transposed."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from oracle import marlin_oracle as mo
from sonar_amd import marlin_linear as ml
from sonar_amd import marlin_utils as mu
from sonar_amd.scalar_type import scalar_types

SQUARE = [(1024, 128, 64), (2048, 128, 128), (512, 128, 32)]


def _converted(k, n, group, device):
    rng = np.random.default_rng(k + n)
    q = rng.integers(0, 16, size=(k, n), dtype=np.int32)
    z = rng.integers(0, 16, size=(k // group, n), dtype=np.int32)
    layer = SimpleNamespace(qweight=torch.from_numpy(mo.awq_pack(q)).to(device), qzeros=torch.from_numpy(mo.awq_pack(z)).to(device),
                            scales=torch.rand(k // group, n).to(torch.float16).to(device), bias=None)
    ml.convert_awq_to_standard_format(layer)
    config = ml.MPLinearLayerConfig((k, n), (k, n), scalar_types.uint4, torch.float16, group, True, False)
    return layer, ml.MarlinLinearKernel(config), mu.marlin_zero_points(torch.from_numpy(z), k // group, n, 4)


@pytest.mark.parametrize("k,n,group", SQUARE + [(1024, 256, 64), (256, 192, 64)])
def test_orientation(k, n, group):
    layer, kernel, want = _converted(k, n, group, "cpu")
    groups = k // group
    assert ml._zero_points_are_transposed(layer.qzeros, layer.scales, groups, n)
    assert torch.equal(kernel._zero_points_by_torch(layer.qzeros.t().contiguous(), n, k, n, k, False), want)
    # without a mark a tensor that fits both ways lies as the scales do: (G, N/8) in GPTQ's layout, (N/8, G) beside (N, G)
    plain = torch.empty((groups, n // 8), dtype=torch.int32)
    assert not ml._zero_points_are_transposed(plain, layer.scales, groups, n)
    assert ml._zero_points_are_transposed(plain.t().contiguous(), layer.scales.t().contiguous(), groups, n)
    plain.input_dim, plain.output_dim = 0, 1
    assert not ml._zero_points_are_transposed(plain, layer.scales.t().contiguous(), groups, n)


@pytest.mark.gpu
@pytest.mark.parametrize("one_launch", [True, False])
@pytest.mark.parametrize("k,n,group", SQUARE + [(8192, 1024, 64)])
def test_loading(k, n, group, one_launch):
    layer, kernel, want = _converted(k, n, group, "cuda:0")
    if not one_launch:
        kernel.workspace = mu.marlin_make_workspace_new(torch.device("cuda:0"))
    assert kernel._load_in_one_launch(layer) == one_launch
    if not one_launch:
        kernel.process_weights_after_loading(layer)
    assert torch.equal(layer.qzeros.cpu(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("k,n,group", [(2048, 128, 128), (512, 128, 32), (4096, 256, 128), (256, 192, 64)])
def test_compressed_tensors_layout(k, n, group):
    """(N, K/8) codes, (N, G) scales and (N/8, G) zero points, without marks: loaded as the same tensors in GPTQ's layout are.
    (Where K/8 == N the codes need marks: a square tensor of codes is (K/8, N).)"""
    other, _, want = _converted(k, n, group, "cuda:0")
    config = ml.MPLinearLayerConfig((k, n), (k, n), scalar_types.uint4, torch.float16, group, True, False)
    gptq = SimpleNamespace(**{**vars(other), "qzeros": other.qzeros.t().contiguous()})
    packed = SimpleNamespace(qweight=other.qweight.t().contiguous(), scales=other.scales.t().contiguous(), bias=None,
                             qzeros=other.qzeros.clone())   # (a clone has no marks)
    for layer in (gptq, packed):
        ml.MarlinLinearKernel(config).process_weights_after_loading(layer)
    assert torch.equal(gptq.qzeros.cpu(), want)
    for name in ("qweight", "scales", "qzeros"):
        assert torch.equal(getattr(packed, name), getattr(gptq, name)), name
