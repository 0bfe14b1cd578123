"""The kernel between decode and prefill (gemm_mid.hip) in tiles of every number of row blocks; one
child process each, because the switch that forces it is read once per process."""
from __future__ import annotations

import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("row_blocks", ["1", "2", "3", "4", "5", "6", "1,6", "2,3", "4,5"])
def test_tiles_of_every_height_meet_the_oracle(row_blocks):
    env = dict(os.environ, SONAR_MARLIN_MID_ROWS=row_blocks)
    out = subprocess.run([sys.executable, "-u", "-m", "tests.mid_rows_child"], cwd=ROOT, env=env,
                         capture_output=True, text=True, timeout=110)
    assert out.returncode == 0 and "all shapes ok" in out.stdout, out.stdout[-1500:] + out.stderr[-1500:]
