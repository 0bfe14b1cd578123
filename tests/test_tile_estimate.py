"""Host only: the time the dispatcher expects of the tile kernels is that of the launch it would make (sonar_debug_tile_estimate
against sonar_debug_tile_schedule)."""
import numpy as np
import pytest

from sonar_amd import _lib
from tests.test_tile_schedule import _rows


def _price(m, n, k):
    """Microseconds of the launch that is made, by the rule of the estimate: a workgroup's loop and what is around it, rounds
    of 256 workgroups, and the sum of the partial tiles.  None: more tiles than compute units, or not the tile kernels'."""
    rows = _rows("sonar_debug_tile_schedule", m, n, k, k // 128)
    if len(rows) == 0 or len(set(rows[:, 0].tolist())) > 1:
        return None
    tile_rows, steps = int(rows[0, 1]), int((rows[:, 5] - rows[:, 4]).max())
    tiles = -(-m // tile_rows) * -(-n // 256)
    if tiles > 256:
        return None
    unit, splits = (0.58 if tile_rows == 128 else 1.0), len(rows) // tiles
    us = 3.3 + -(-len(rows) // 256) * unit * (1.21 * steps + 11.2)
    return us + 1.1 + 1.24e-6 * splits * m * n if splits > 1 else us


@pytest.mark.parametrize("m", [97, 112, 128])
@pytest.mark.parametrize("n", [16448, 17408, 20480, 28672, 32768])
@pytest.mark.parametrize("k", [1024, 4096, 7168])
def test_97_to_128_rows_on_wide_matrices(m, n, k):
    want = _price(m, n, k)
    assert want is not None
    assert _lib.load().sonar_debug_tile_estimate(m, n, k) == pytest.approx(want, rel=1e-6)


def test_random_shapes():
    rng = np.random.default_rng(3)
    seen = 0
    for _ in range(800):
        m, n, k = int(rng.integers(65, 4000)), 64 * int(rng.integers(1, 300)), 128 * int(rng.integers(1, 100))
        want = _price(m, n, k)
        if want is not None:
            seen += 1
            assert _lib.load().sonar_debug_tile_estimate(m, n, k) == pytest.approx(want, rel=1e-6), (m, n, k)
    assert seen > 200
