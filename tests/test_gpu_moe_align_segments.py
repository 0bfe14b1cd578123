"""Routing of slots by several workgroups, a segment of them each: sizes at the ends of segments (one up to 5000 slots, 1024
slots each up to 65536, more beyond), one expert, uneven experts and the most of one launch, invalid ids, an expert map, and
ids that do not lie at 16 bytes."""
from __future__ import annotations

import pytest
import torch

from sonar_amd import fused_moe

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("numel", [1025, 5000, 5001, 6143, 6145, 65535, 65536, 65537, 131073])
@pytest.mark.parametrize("experts,offset", [(1, 0), (8, 1), (33, 3), (768, 0), (769, 2)])
@pytest.mark.parametrize("mapped", [False, True])
def test_segments(numel, experts, offset, mapped):
    gen = torch.Generator().manual_seed(numel + experts)
    # half of the slots on a few experts, some ids outside the table
    ids = torch.randint(0, experts, (numel,), generator=gen, dtype=torch.int32)
    ids = torch.where(torch.rand(numel, generator=gen) < 0.5, ids // 7, ids)
    ids[torch.rand(numel, generator=gen) < 0.01] = experts
    ids[torch.rand(numel, generator=gen) < 0.01] = -1
    emap = None
    if mapped:
        emap = torch.randperm(experts, generator=gen).to(torch.int32)
        emap[torch.rand(experts, generator=gen) < 0.2] = -1
    want = fused_moe.moe_align_block_size(ids.view(-1, 1), 64, experts, emap, ignore_invalid_experts=True)
    held = torch.zeros(numel + 8, dtype=torch.int32, device=DEV)
    there = held[offset:offset + numel].view(-1, 1)
    there.copy_(ids.view(-1, 1))
    got = fused_moe.moe_align_block_size(there, 64, experts, emap.to(DEV) if mapped else None, ignore_invalid_experts=True)
    for g, w in zip(got, want):
        assert torch.equal(g.cpu(), w)
