"""A grouped call on 64-slot blocks whose routing left no block at all (every expert lives on another rank): nothing is read or
written, with either number of blocks per round of the table kernel."""
import numpy as np
import pytest

from oracle import marlin_oracle as mo
from tests import gpu_util as gu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [300, 9000])
def test_no_block(tokens):
    from tests.test_gpu_moe import Experts, route
    e, top_k, k, n = 4, 2, 256, 128
    ex = Experts(5, e, k, n, 128, "bf16")
    topk_ids, topk_w = route(5, tokens, e, top_k)
    sorted_ids, expert_ids, _ = mo.moe_align_block_size(topk_ids, 64, e)
    a = gu.dev_bits16(mo.make_activations(9, tokens, k, "bf16"), "bf16")
    assert np.all(gu.host_f32(ex.gemm(a, sorted_ids, expert_ids, 0, topk_w, 64, top_k, tokens, False)) == 0.0)
