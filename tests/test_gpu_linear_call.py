"""The one-call linear op against the steps it stands for, and the quantisation of its activations where the
eight-column loads begin, end and do not apply."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import marlin_oracle as mo
from sonar_amd import marlin_utils as mu
from sonar_amd import ops
from sonar_amd.scalar_type import scalar_types

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols,stride", [(8, 8), (2040, 2040), (2048, 2056), (2056, 2060), (513, 513), (16384, 16384), (18440, 18440)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_quantised_activations_match_the_oracle(cols, stride, dtype):
    x = (torch.randn((3, stride), device="cuda") * 3).to(dtype)[:, :cols]
    x[2] = 0
    q, s = ops.per_token_quant_int8(x)
    want_q, want_s = mo.per_token_quant_int8(x.float().cpu().numpy())
    assert np.array_equal(q.cpu().numpy(), want_q) and np.array_equal(s.cpu().numpy(), want_s)
    f, fs = ops.per_token_quant_fp8(x)
    host = x.float().cpu()
    scale = (host.abs().amax(1, keepdim=True) / 448.0).clamp_min(1.0 / (448.0 * 512.0))
    want_f = (host * (1.0 / scale)).clamp(-448, 448).to(torch.float8_e4m3fn)
    assert torch.equal(fs.cpu(), scale) and torch.equal(f.view(torch.uint8).cpu(), want_f.view(torch.uint8))


@pytest.mark.parametrize("shape,act", [((5,), None), ((2, 3), None), ((), None), ((4,), torch.int8), ((2, 2), torch.float8_e4m3fn)])
@pytest.mark.parametrize("n,k", [(256, 512), (192, 480)])
def test_linear_call_is_pad_quantise_multiply_unpad(shape, act, n, k):
    padded_n, padded_k = (n + 63) // 64 * 64, (k + 127) // 128 * 128
    gen = torch.Generator(device="cuda").manual_seed(3)
    weight = torch.randint(-2 ** 31, 2 ** 31 - 1, (padded_k // 16, 2 * padded_n), dtype=torch.int32, device="cuda", generator=gen)
    scales = (torch.rand((1, padded_n), device="cuda", generator=gen) * 1e-2).half()
    x = torch.randn(shape + (k,), device="cuda", generator=gen).half()
    factor = torch.tensor([0.37], device="cuda") if act == torch.int8 else None
    bias = torch.randn(padded_n, device="cuda", generator=gen).half()
    empty = torch.empty(0, dtype=torch.int32, device="cuda")
    workspace = mu.marlin_make_workspace_new(torch.device("cuda"))
    got = mu.apply_gptq_marlin_linear(x, weight, scales, empty, empty, empty, workspace, scalar_types.uint4b8, n, k, True,
                                      factor, bias, True, act)
    a = mu.marlin_pad_dim(x.reshape(-1, k), k, padded_k)
    a_scales = None
    if act is not None:
        a, a_scales = mu.marlin_quant_input(a, act)
        if factor is not None:
            a_scales = a_scales * factor
    want = ops.marlin_gemm(a, None, weight, bias, scales, a_scales, None, empty, empty, empty, workspace,
                           scalar_types.uint4b8, a.shape[0], padded_n, padded_k, True, False, True, False)
    assert got.shape == shape + (n,) and got.is_contiguous()
    assert torch.equal(got.reshape(-1, n), want[:, :n])


# what a product with the (rows, 1) scales of the activations takes
@pytest.mark.parametrize("factor", [
    lambda: torch.tensor(0.37), lambda: 0.37, lambda: torch.tensor([0.37], device="cuda"), lambda: torch.tensor(0.37, device="cuda"),
    lambda: torch.tensor([0.37], device="cuda").half(), lambda: torch.tensor(0.37, device="cuda", dtype=torch.float64),
    lambda: torch.linspace(0.2, 0.9, 5, device="cuda").unsqueeze(1), lambda: torch.full((1, 1), 0.37, device="cuda"),
], ids=["cpu", "number", "float", "scalar", "half", "double_scalar", "per_row", "matrix"])
def test_factor_of_the_activation_scales_in_every_form(factor):
    m, n, k = 5, 128, 256
    gen = torch.Generator(device="cuda").manual_seed(4)
    weight = torch.randint(-2 ** 31, 2 ** 31 - 1, (k // 16, 2 * n), dtype=torch.int32, device="cuda", generator=gen)
    scales = (torch.rand((1, n), device="cuda", generator=gen) * 1e-2).half()
    x = torch.randn((m, k), device="cuda", generator=gen).half()
    empty = torch.empty(0, dtype=torch.int32, device="cuda")
    workspace = mu.marlin_make_workspace_new(torch.device("cuda"))
    got = mu.apply_gptq_marlin_linear(x, weight, scales, empty, empty, empty, workspace, scalar_types.uint4b8, n, k, True,
                                      factor(), None, True, torch.int8)
    a, a_scales = mu.marlin_quant_input(x, torch.int8)
    want = ops.marlin_gemm(a, None, weight, None, scales, a_scales * factor(), None, empty, empty, empty, workspace,
                           scalar_types.uint4b8, m, n, k, True, False, True, False)
    assert torch.equal(got, want)
