"""The W4A8 kernel of gemm_a8_block.hip in each of its tiles, with K in one piece and split over workgroups; one
child process each, because the switch that forces the tile is read once per process."""
from __future__ import annotations

import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("shape", ["1,4,1", "1,4,3", "2,4,1", "3,2,1", "3,1,1", "3,1,2", "4,1,1"])
def test_every_tile_meets_the_oracle(shape):
    env = dict(os.environ, SONAR_MARLIN_A8_SHAPE=shape)
    out = subprocess.run([sys.executable, "-u", "-m", "tests.a8_block_child"], cwd=ROOT, env=env,
                         capture_output=True, text=True, timeout=110)
    assert out.returncode == 0 and "all shapes ok" in out.stdout, out.stdout[-1500:] + out.stderr[-1500:]
