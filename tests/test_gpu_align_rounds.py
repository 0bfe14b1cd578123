"""moe_align_block_size around the number of slots that a wavefront of its kernel reads at a time: one round of 64, up to eight,
more, with a last round that is not full, slots without an expert, and more experts than one launch places."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from sonar_amd import fused_moe
from tests import gpu_util as gu
from tests import test_gpu_moe as tm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,e", [(1023, 5), (1024, 5), (1025, 5), (8191, 16), (8192, 16), (8193, 16), (40001, 64), (9000, 769)])
def test_rounds_of_slots(m, e):
    tm.test_moe_align_kernel_matches_oracle(m, 1, e, 64)


@pytest.mark.parametrize("m", [900, 5000, 20000])
def test_rounds_of_slots_with_an_expert_map(m):
    rng = np.random.default_rng(m)
    e = 24
    ids = torch.from_numpy(rng.integers(0, e, size=(m, 1), dtype=np.int32))
    emap = torch.from_numpy(np.where(np.arange(e) % 3 == 0, -1, rng.permutation(e)).astype(np.int32))
    for ignore in (True, False):
        want = fused_moe.moe_align_block_size(ids, 64, e, emap, ignore_invalid_experts=ignore)        # CPU: torch
        got = fused_moe.moe_align_block_size(ids.to(gu.DEV), 64, e, emap.to(gu.DEV), ignore_invalid_experts=ignore)
        past = int(want[2][0])
        assert int(got[2][0]) == past
        assert torch.equal(got[0].cpu()[:past], want[0][:past]) and torch.equal(got[1].cpu(), want[1])
