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
def test_general_path(k, n, group):
    layer, kernel, want = _converted(k, n, group, "cpu")
    assert torch.equal(kernel._zero_points_by_torch(layer.qzeros, n, k, n, k, False), want)
    # without a mark a tensor that fits both ways is (G, N/8), as before there was one
    plain = mu.pack_cols(torch.arange(k // group * n, dtype=torch.int32).reshape(k // group, n) % 16, 4, k // group, n)
    codes = mu.unpack_cols(plain, 4, k // group, n)
    assert torch.equal(kernel._zero_points_by_torch(plain, n, k, n, k, False), mu.marlin_zero_points(codes, k // group, n, 4))


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
