"""Kernels that wait for memory operations with hand-counted `s_waitcnt vmcnt(N)` must not spill: a spill's
own loads and stores would count too and weaken those waits.  Read from the metadata of the built library."""
from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin"


@pytest.mark.parametrize("kernel,at_least", [
    ("marlin_mid_gemm", 140), ("marlin_a8_block", 50), ("marlin_stream_fast_kernel", 80), ("marlin_tile_async_kernel", 10),
    ("marlin_tile_wide_kernel", 30), ("marlin_tile_wide_pair_kernel", 20), ("marlin_tile_twin_kernel", 18)])
def test_hand_counted_kernels_do_not_spill(kernel, at_least, tmp_path):
    from sonar_amd import _lib
    _lib.load()
    if not os.path.exists(f"{LLVM}/llvm-objdump"):
        pytest.skip("llvm-objdump not available")
    lib = shutil.copy(_lib.lib_path(), tmp_path)
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", lib], cwd=tmp_path, capture_output=True, check=True, timeout=60)
    seen = 0
    for obj in tmp_path.glob("*gfx950*"):
        notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", str(obj)], capture_output=True, text=True, timeout=60)
        for m in re.finditer(r"\.name:\s+(\S+).*?\.private_segment_fixed_size:\s+(\d+).*?\.vgpr_spill_count:\s+(\d+)",
                             notes.stdout, re.S):
            if kernel in m.group(1):
                seen += 1
                assert m.group(2) == "0" and m.group(3) == "0", f"{m.group(1)}: scratch {m.group(2)}, spills {m.group(3)}"
    assert seen >= at_least, f"{seen} forms of {kernel} in the library"
