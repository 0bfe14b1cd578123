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


# us in marlin_mid_gemm and in the tile kernels: one of the two at least a sixth faster
@pytest.mark.parametrize("code,dtype,group,m,k,n,mid,tile", [
    ("fp8", "bf16", -1, 271, 6144, 6400, 34.9, 51.2), ("fp8", "bf16", -1, 134, 3968, 26240, 53.0, 70.5),
    ("fp8", "bf16", -1, 504, 4480, 2752, 25.9, 34.4), ("fp8", "bf16", -1, 1270, 6656, 1472, 34.9, 46.4),
    ("fp8", "bf16", -1, 818, 3840, 5376, 51.9, 67.4), ("fp8", "bf16", -1, 274, 8832, 15104, 97.8, 129.1),
    ("uint8b128", "bf16", -1, 196, 1664, 11392, 24.0, 31.2), ("uint8b128", "bf16", -1, 123, 8832, 16128, 42.5, 48.9),
    ("uint8b128", "bf16", -1, 207, 7296, 8448, 39.3, 49.3), ("uint8b128", "bf16", -1, 125, 13440, 17472, 104.8, 77.2),
    ("uint8b128", "fp16", 128, 122, 13056, 22016, 130.6, 104.7), ("uint8b128", "fp16", 128, 203, 4352, 10688, 28.7, 37.7),
    ("uint4", "fp16", 64, 113, 6656, 16640, 60.8, 45.1), ("uint4b8", "bf16", -1, 187, 5888, 10304, 30.7, 44.7)])
def test_choice_between_the_mid_size_and_the_tile_kernels(code, dtype, group, m, k, n, mid, tile):
    types = {"fp8": _lib.TYPE_FLOAT8_E4M3FN, "uint8b128": _lib.TYPE_UINT8B128, "uint4": _lib.TYPE_UINT4, "uint4b8": _lib.TYPE_UINT4B8}
    dtypes = {"fp16": _lib.DTYPE_F16, "bf16": _lib.DTYPE_BF16}
    chosen = _lib.load().sonar_debug_mid_beats_tiles(m, n, k, 1 if group == -1 else k // group, dtypes[dtype], types[code])
    assert chosen == int(mid < tile)
