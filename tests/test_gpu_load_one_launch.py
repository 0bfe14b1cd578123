"""A 4-bit projection loaded by one launch: the same bytes as the general path (taken here by a kernel object that already
holds a workspace), over groups, zero-point layouts and sizes whose last workgroup of each kind is ragged."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _layer(k, n, group, dtype, zeros, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    groups = 1 if group == -1 else k // group

    def words(rows, cols):
        return torch.randint(-2 ** 31, 2 ** 31 - 1, (rows, cols), dtype=torch.int32, device=DEV, generator=gen)
    layer = SimpleNamespace(qweight=words(k // 8, n), scales=torch.rand(groups, n, device=DEV, generator=gen).to(dtype),
                            bias=torch.rand(n, device=DEV, generator=gen).to(dtype))
    if zeros:
        layer.qzeros = words(n // 8, groups) if zeros == "transposed" else words(groups, n // 8)
    return layer


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("zeros", [None, "rows", "transposed"])
@pytest.mark.parametrize("k,n,group", [(128, 64, -1), (128, 64, 128), (128, 192, 32), (256, 16384, 128), (384, 1088, 64),
                                       (1152, 2112, 128), (1024, 64, 64)])
def test_same_as_the_general_path(k, n, group, zeros, dtype):
    from sonar_amd import marlin_linear as ml
    from sonar_amd.scalar_type import scalar_types
    cfg = ml.MPLinearLayerConfig((k, n), (k, n), scalar_types.uint4 if zeros else scalar_types.uint4b8, dtype, group,
                                 bool(zeros), False)
    one, general = (_layer(k, n, group, dtype, zeros, k + n) for _ in range(2))
    kernels = [ml.MarlinLinearKernel(cfg) for _ in range(2)]
    kernels[1].workspace = torch.ones(torch.cuda.get_device_properties(0).multi_processor_count, dtype=torch.int32,
                                      device=DEV)
    raw = one.qweight
    assert kernels[0]._load_in_one_launch(one)
    kernels[1].process_weights_after_loading(general)
    assert one.qweight is not raw and vars(one).keys() == vars(general).keys()
    for name, value in vars(general).items():
        if value is None:
            assert getattr(one, name) is None
            continue
        mine = getattr(one, name)
        assert mine.shape == value.shape and mine.dtype == value.dtype and mine.stride() == value.stride(), name
        assert isinstance(mine, torch.nn.Parameter) == isinstance(value, torch.nn.Parameter), name
        assert torch.equal(mine, value), name
    a, b = kernels[0].workspace, kernels[1].workspace
    assert a.shape == b.shape and a.dtype == b.dtype and a.device == b.device and int(a.abs().sum()) == 0
    assert kernels[0].is_k_full == kernels[1].is_k_full


def test_other_tensors_take_the_general_path():
    from sonar_amd import marlin_linear as ml
    from sonar_amd.scalar_type import scalar_types
    k, n, group = 256, 192, 64

    def refused(change, **over):
        cfg = ml.MPLinearLayerConfig((k, n), (k, n), **{**dict(weight_type=scalar_types.uint4b8, act_type=torch.float16,
                                                              group_size=group, zero_points=False, has_g_idx=False), **over})
        layer = _layer(k, n, group, torch.float16, None, 1)
        change(layer)
        before = dict(vars(layer))
        assert not ml.MarlinLinearKernel(cfg)._load_in_one_launch(layer)
        assert all(getattr(layer, name) is value for name, value in before.items())

    def put(name, make):
        return lambda layer: setattr(layer, name, make(getattr(layer, name)))
    refused(put("scales", lambda s: s.float()))
    refused(put("scales", lambda s: s.t().contiguous()))
    refused(put("scales", lambda s: torch.nn.Parameter(s)))
    refused(put("scales", lambda s: torch.cat([s, s], 1)[:, :n]))
    refused(put("qweight", lambda q: q.t().contiguous()))
    refused(put("qweight", lambda q: q.cpu()))
    refused(put("qweight", lambda q: torch.cat([q, q], 1)[:, :n]))
    refused(lambda layer: None, act_type=torch.int8)
    refused(lambda layer: setattr(layer, "qzeros", torch.zeros(k // group, n, dtype=torch.int32, device=DEV)),
            weight_type=scalar_types.uint4, zero_points=True)

    def marked(layer):
        layer.qweight.input_dim = 1
    refused(marked)


def test_opcheck():
    k, n, groups = 256, 192, 4
    layer = _layer(k, n, k // groups, torch.bfloat16, "rows", 3)
    for zeros, transposed in ((None, False), (layer.qzeros, False), (layer.qzeros.t().contiguous(), True)):
        torch.library.opcheck(torch.ops.sonar_amd.load_gptq_linear, (layer.qweight, layer.scales, zeros, True, transposed))
    for bad in (layer.scales.float(), layer.scales[:, :128], layer.scales.cpu()):
        with pytest.raises(RuntimeError):
            torch.ops.sonar_amd.load_gptq_linear(layer.qweight, bad, None, True, False)
    with pytest.raises(RuntimeError):
        torch.ops.sonar_amd.load_gptq_linear(layer.qweight, layer.scales, layer.qzeros[:2], True, False)
    with pytest.raises(RuntimeError):   # N is no multiple of 64
        torch.ops.sonar_amd.load_gptq_linear(layer.qweight[:, :96].contiguous(), layer.scales[:, :96].contiguous(), None,
                                             True, False)


@pytest.mark.parametrize("k", [1, 63, 64, 65, 128, 1000, 1024, 4096, 14336, 32768])
@pytest.mark.parametrize("kind", ["groups", "descending", "any"])
def test_sorted_group_indices(k, kind):
    from sonar_amd.marlin_utils import marlin_sort_g_idx
    gen = torch.Generator().manual_seed(k)
    g_idx = {"groups": lambda: (torch.arange(k) // 128)[torch.randperm(k, generator=gen)],
             "descending": lambda: torch.arange(k).flip(0),
             "any": lambda: torch.randint(-2 ** 31, 2 ** 31 - 1, (k,), generator=gen)
             .where(torch.rand(k, generator=gen) < 0.5, torch.tensor(-2 ** 31))}[kind]().to(torch.int32)
    order = torch.argsort(g_idx, stable=True).to(torch.int32)
    got, got_order = marlin_sort_g_idx(g_idx.to(DEV))
    assert got.dtype == got_order.dtype == torch.int32
    assert torch.equal(got_order.cpu(), order) and torch.equal(got.cpu(), g_idx[order.long()])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("k,n,group,full_k", [(128, 64, 128, 128), (128, 192, 32, 128), (384, 1088, 64, 768), (1152, 2112, 128, 1152),
                                              (4096, 64, -1, 4096)])
def test_act_order_same_as_the_general_path(k, n, group, full_k, dtype):
    from sonar_amd import marlin_linear as ml
    from sonar_amd.scalar_type import scalar_types
    cfg = ml.MPLinearLayerConfig((full_k, n), (k, n), scalar_types.uint4b8, dtype, group, False, True)
    one, general = (_layer(k, n, group, dtype, None, k + n) for _ in range(2))
    groups = torch.arange(k, dtype=torch.int32, device=DEV) // (k if group == -1 else group)
    shuffled = groups[torch.randperm(k, device=DEV, generator=torch.Generator(device=DEV).manual_seed(5))]
    kernels = [ml.MarlinLinearKernel(cfg) for _ in range(2)]
    for layer in (one, general):
        layer.g_idx = torch.nn.Parameter(shuffled.clone(), requires_grad=False)
    kernels[1].workspace = torch.ones(torch.cuda.get_device_properties(0).multi_processor_count, dtype=torch.int32, device=DEV)
    assert kernels[0]._load_in_one_launch(one) and not kernels[1]._load_in_one_launch(general)
    kernels[1].process_weights_after_loading(general)
    assert vars(one).keys() == vars(general).keys() and kernels[0].is_k_full == kernels[1].is_k_full == (k == full_k)
    for name, value in vars(general).items():
        mine = getattr(one, name)
        assert type(mine) is type(value), name
        assert value is None or (mine.dtype == value.dtype and mine.stride() == value.stride() and torch.equal(mine, value)), name
    assert int(kernels[0].workspace.abs().sum()) == 0
    torch.library.opcheck(torch.ops.sonar_amd.sort_g_idx, (shuffled,))
    raw = _layer(k, n, group, dtype, None, 1)
    torch.library.opcheck(torch.ops.sonar_amd.load_gptq_act_order, (raw.qweight, raw.scales, shuffled, group != -1))
    # a layer that holds its order already keeps that tensor, on the general path
    again, held = _layer(k, n, group, dtype, None, k + n), torch.zeros(k, dtype=torch.int32, device=DEV)
    again.g_idx, again.g_idx_sort_indices = shuffled, held
    ml.MarlinLinearKernel(cfg).process_weights_after_loading(again)
    assert again.g_idx_sort_indices is held and torch.equal(held, general.g_idx_sort_indices) and torch.equal(again.qweight, one.qweight)
    for bad in (shuffled[:-1], shuffled.long(), shuffled.cpu()):
        with pytest.raises(RuntimeError):
            torch.ops.sonar_amd.load_gptq_act_order(raw.qweight, raw.scales, bad, group != -1)
