"""Host only: launches of the grouped wide kernel with both tile sizes, from the library's own planning and mapping code
(sonar_debug_moe_pair_schedule): every tile and K step once, within the scratch that the partial tiles have."""
import ctypes

import numpy as np
import pytest

from sonar_amd import _lib


def _schedule(big, small, max_row_tiles, n, k, with_partial):
    lib = _lib.load()
    chosen = (ctypes.c_int32 * 3)()
    args = (big, small, max_row_tiles, n, k, with_partial, chosen)
    count = lib.sonar_debug_moe_pair_schedule(*args, None, 0)
    assert count >= 0
    out = np.zeros((max(count, 1), 6), dtype=np.int32)
    assert lib.sonar_debug_moe_pair_schedule(*args, out.ctypes.data_as(ctypes.c_void_p), count) == count
    return list(chosen), out[:count]


def _check(big, small, max_row_tiles, n, k, with_partial):
    (halved, *splits), rows = _schedule(big, small, max_row_tiles, n, k, with_partial)
    tiles_n, steps = (n + 255) // 256, k // 64
    assert 0 <= halved <= big
    for size, tiles_m, asked in ((256, big - halved, splits[0]), (128, small + 2 * halved, splits[1])):
        mine = rows[rows[:, 1] == size]
        seen = {}
        for _, _, tm, tn, k0, k1 in mine.tolist():
            assert 0 <= tm < tiles_m and 0 <= tn < tiles_n and 0 <= k0 < k1 <= steps
            seen.setdefault((tm, tn), []).append((k0, k1))
        assert len(seen) == tiles_m * tiles_n
        for ranges in seen.values():
            ranges.sort()
            assert ranges[0][0] == 0 and ranges[-1][1] == steps and len(ranges) <= asked
            assert all(a[1] == b[0] for a, b in zip(ranges, ranges[1:]))
        if asked > 1:
            assert with_partial and k % 256 == 0 and tiles_m * tiles_n <= 128 and len(mine) <= 256
    return halved, splits


@pytest.mark.parametrize("k,n", [(4096, 28672), (14336, 4096), (1024, 320), (2880, 5760), (64, 256), (768, 1280)])
def test_every_tile_and_k_step_once(k, n):
    for with_partial in (0, 1):
        for big, small in ((0, 0), (0, 1), (1, 0), (2, 3), (8, 8), (9, 0), (32, 4), (40, 17), (0, 64), (100, 3)):
            _check(big, small, 4 * big + 2 * small + 3, n, k, with_partial)


def test_random_launches():
    rng = np.random.default_rng(5)
    halved = cut = 0
    for _ in range(300):
        big, small = int(rng.integers(0, 40)), int(rng.integers(0, 40))
        n, k = 64 * int(rng.integers(1, 80)), 64 * int(rng.integers(1, 257))
        h, splits = _check(big, small, 4 * big + 2 * small, n, k, int(rng.integers(0, 2)))
        halved += h > 0
        cut += max(splits) > 1
    assert halved > 20 and cut > 5


def test_arguments_out_of_range():
    lib = _lib.load()
    chosen = (ctypes.c_int32 * 3)()
    assert lib.sonar_debug_moe_pair_schedule(2, 1, 6, 256, 256, 0, chosen, None, 0) == -1
    assert lib.sonar_debug_moe_pair_schedule(1, 1, 8, 256, 100, 0, chosen, None, 0) == -1
