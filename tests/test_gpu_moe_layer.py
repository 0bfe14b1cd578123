"""Routing kernels at the edges of their launches, and the one-call layer against the layer run op by op."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# one slot, shares that end inside a round of 64 slots, 768 experts (the last count with one launch) and 769
@pytest.mark.parametrize("tokens,top_k,experts,block", [(1, 1, 1, 8), (1, 8, 64, 8), (65, 2, 8, 16), (1023, 1, 3, 64),
                                                        (2049, 4, 32, 64), (700, 8, 768, 16), (700, 8, 769, 16),
                                                        (9001, 8, 256, 64)])
@pytest.mark.parametrize("mapped", [False, True])
def test_align_block_size_matches_the_torch_form(tokens, top_k, experts, block, mapped):
    from sonar_amd import fused_moe
    gen = torch.Generator().manual_seed(tokens + experts)
    ids = torch.rand((tokens, experts), generator=gen).topk(min(top_k, experts), dim=1).indices.to(torch.int32)
    ids[0, 0] = experts + 5    # a slot that belongs to nobody
    emap = None
    if mapped:
        emap = torch.full((experts,), -1, dtype=torch.int32)
        emap[::2] = torch.arange((experts + 1) // 2, dtype=torch.int32)
    want = fused_moe.moe_align_block_size(ids, block, experts, emap, ignore_invalid_experts=True)
    got = fused_moe.moe_align_block_size(ids.to(DEV), block, experts, None if emap is None else emap.to(DEV),
                                         ignore_invalid_experts=True)
    for g, w in zip(got, want):
        assert torch.equal(g.cpu(), w)


def _layer(experts, hidden, inter, dtype, zeros=False):
    gen = torch.Generator(device=DEV).manual_seed(experts * hidden + inter)

    def words(*shape):
        return torch.randint(-2 ** 31, 2 ** 31 - 1, shape, dtype=torch.int32, device=DEV, generator=gen)

    def scales(*shape):
        return (torch.rand(shape, device=DEV, generator=gen) * 9e-3 + 1e-3).to(dtype)
    w = dict(w1=words(experts, hidden // 16, 4 * inter), w2=words(experts, inter // 16, 2 * hidden),
             w1_scale=scales(experts, hidden // 128, 2 * inter), w2_scale=scales(experts, inter // 128, hidden))
    if zeros:
        w.update(w1_zeros=words(experts, hidden // 128, inter // 4), w2_zeros=words(experts, inter // 128, hidden // 8))
    return w, gen


def _run(w, x, tw, ti, **kw):
    from sonar_amd import fused_moe
    from sonar_amd.scalar_type import scalar_types
    wtype = scalar_types.uint4 if "w1_zeros" in w else scalar_types.uint4b8
    return fused_moe.fused_marlin_moe(x, w["w1"], w["w2"], None, None, w["w1_scale"], w["w2_scale"], tw, ti, wtype.id,
                                      w1_zeros=w.get("w1_zeros"), w2_zeros=w.get("w2_zeros"), **kw)


@pytest.mark.parametrize("tokens,top_k,experts", [(1, 2, 8), (5, 8, 64), (100, 2, 4), (600, 4, 8)])
@pytest.mark.parametrize("activation", ["silu", "swigluoai", "gelu"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_one_call_is_the_layer_op_by_op(tokens, top_k, experts, activation, dtype):
    from sonar_amd import fused_moe
    w, gen = _layer(experts, 256, 384, dtype, zeros=activation == "gelu")
    x = torch.randn((tokens, 256), device=DEV, generator=gen).to(dtype)
    tw, ti = torch.rand((tokens, experts), device=DEV, generator=gen).topk(top_k, dim=1)
    by_op = _run(w, x, tw, ti, activation=activation, moe_sum=lambda y, out, ids, emap: fused_moe.moe_sum(y, out))
    assert torch.equal(_run(w, x, tw, ti, activation=activation), by_op)
    given = torch.empty_like(x)
    caches = dict(intermediate_cache13=torch.empty(tokens * top_k * 768 + 8, dtype=dtype, device=DEV),
                  intermediate_cache2=torch.empty((tokens * top_k + 1, 384), dtype=dtype, device=DEV))
    assert _run(w, x, tw, ti, activation=activation, output=given, **caches) is given and torch.equal(given, by_op)


def test_more_blocks_than_the_tile_table_has_threads():
    """1125 and more blocks of 64 slots: the table is built in two rounds; tokens do not depend on each other."""
    w, gen = _layer(8, 128, 128, torch.bfloat16)
    x = torch.randn((9000, 128), device=DEV, generator=gen).to(torch.bfloat16)
    tw, ti = torch.rand((9000, 8), device=DEV, generator=gen).topk(8, dim=1)
    whole = _run(w, x, tw, ti).float()
    parts = torch.cat([_run(w, x[i:i + 900], tw[i:i + 900], ti[i:i + 900]) for i in range(0, 9000, 900)]).float()
    assert (whole - parts).norm() <= 5e-3 * parts.norm()
