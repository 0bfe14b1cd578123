"""128-row tiles two at a time on a compute unit (marlin_tile_twin_kernel): which dense calls have them and that their tiles cover C
once; that the compiler left the accumulators where the loop's instructions have them; every form against the oracle at the edges of
its tiles and steps; and, with the tile kernels that would run otherwise in another process, the same bits from dense calls and from
mixture-of-experts layers."""
from __future__ import annotations

import hashlib
import os
import re
import shutil
import subprocess
import sys

import pytest
import torch

from sonar_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = "cuda:0"


@pytest.mark.parametrize("m,k,n,groups,dtype,fp4,twin", [
    (2100, 192, 7360, 3, "fp16", 0, True), (332, 3200, 17728, 25, "fp16", 0, True), (855, 1024, 17472, 32, "bf16", 1, True),
    (8000, 1024, 11008, 8, "bf16", 0, True), (2100, 64, 7360, 2, "fp16", 0, True),
    (4000, 7168, 11008, 56, "bf16", 0, False),     # a long K in bf16
    (4096, 4096, 4096, 32, "fp16", 0, False),      # one round of 256-row tiles
    (1000, 1024, 4096, 8, "fp16", 0, False),       # few tiles
    (2100, 192, 7360, 1, "fp16", 0, False)])       # one group
def test_which_calls_and_what_their_tiles_cover(m, k, n, groups, dtype, fp4, twin):
    from tests.test_tile_schedule import _check_cover, _rows
    rows = _rows("sonar_debug_twin_schedule", m, n, k, groups, _lib.DTYPE_F16 if dtype == "fp16" else _lib.DTYPE_BF16, fp4)
    assert (len(rows) > 0) == twin
    if twin:
        _check_cover(rows, {128: set(range(-(-m // 128)))}, -(-n // 256), k // 64)


@pytest.mark.parametrize("rows,slots,k,twin", [
    (1 << 19, (1 << 19) + 64, 2048, True), (1 << 20, (1 << 20) + 64, 2048, False),
    (1 << 20, 64 * 8, 2048, False),       # few slots given, whose ids reach rows of A behind the first 4 GiB
    ((1 << 20) - 1, 64 * 8, 2048, True),  # (the last row ends there)
    (1000, 1 << 20, 2048, False)])        # many slots of few rows: a copy of A by slot
def test_rows_of_a_lie_within_32_bits(rows, slots, k, twin):
    assert _lib.load().sonar_debug_moe_twin(rows, slots, 8, 4096, k, k // 64, _lib.DTYPE_F16, 0, 0) == twin


def test_accumulators_stay_in_place(tmp_path):
    """The matrix instructions are asm statements, around which the compiler pads no hazard: an accumulator that it moved out of its
    registers around the loop would be read before the last sums have arrived."""
    llvm = "/opt/rocm/llvm/bin"
    _lib.load()
    if not os.path.exists(f"{llvm}/llvm-objdump"):
        pytest.skip("llvm-objdump not available")
    lib = shutil.copy(_lib.lib_path(), tmp_path)
    subprocess.run([f"{llvm}/llvm-objdump", "--offloading", lib], cwd=tmp_path, capture_output=True, check=True, timeout=60)
    seen = 0
    for obj in tmp_path.glob("*gfx950*"):
        names = subprocess.run([f"{llvm}/llvm-readelf", "--symbols", "--wide", str(obj)], capture_output=True, text=True, timeout=60).stdout
        names = {w for w in re.findall(r"\S*marlin_tile_twin_kernel\S*", names) if not w.endswith(".kd")}
        if not names:
            continue
        asm = subprocess.run([f"{llvm}/llvm-objdump", "-d", "--mcpu=gfx950", "--no-show-raw-insn",
                              "--disassemble-symbols=" + ",".join(sorted(names)), str(obj)], capture_output=True, text=True, timeout=300).stdout
        seen += len(re.findall(r"<\S*marlin_tile_twin_kernel\S*>:", asm))
        assert not re.search(r"v_accvgpr_write|v_accvgpr_mov|scratch_", asm)
    assert seen >= 18


def _child(what: str, *args: str, **env: str) -> str:
    out = subprocess.run([sys.executable, "-u", "-m", "tests.test_twin_tiles", what, *args], cwd=ROOT, capture_output=True, text=True,
                         env=dict(os.environ, **env), timeout=110)
    assert out.returncode == 0 and out.stdout.strip().endswith("done"), out.stdout[-1500:] + out.stderr[-1500:]
    return out.stdout


# (the mid-size kernel would take some of these sizes)
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
def test_dense_forms_against_the_oracle(dtype):
    _child("oracle", dtype, SONAR_MARLIN_NO_MID="1")


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["dense", "layers"])
def test_same_bits_as_the_other_tile_kernels(what):
    assert _child(what, SONAR_MARLIN_NO_MID="1") == _child(what, SONAR_MARLIN_NO_MID="1", SONAR_MARLIN_NO_TWIN_TILES="1")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
def test_the_other_tile_kernels_on_these_sizes(dtype):
    out = subprocess.run([sys.executable, "-u", "-m", "tests.test_gpu_two_tile_sizes", dtype], cwd=ROOT, capture_output=True, text=True,
                         env=dict(os.environ, SONAR_MARLIN_NO_MID="1", SONAR_MARLIN_NO_TWIN_TILES="1"), timeout=110)
    assert out.returncode == 0 and "all forms ok" in out.stdout, out.stdout[-1500:] + out.stderr[-1500:]
    _child("grouped", dtype, SONAR_MARLIN_NO_TWIN_TILES="1")


# 256-row tiles of groups of 32 rows: 252 tiles, a launch of that size alone, in front of which these tiles stand for most calls
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
def test_256_row_tiles_of_small_groups(dtype):
    _child("small_groups", dtype, SONAR_MARLIN_NO_MID="1", SONAR_MARLIN_NO_TWIN_TILES="1")


def _small_groups(dtype: str) -> None:
    from tests import gpu_util as gu
    from tests import test_gpu_parity as tp
    for k, zp in ((192, False), (128, True)):
        tp.test_wide_tile_kernel_forms_within_tolerance(gu, dtype, 2049, k, 7168, 32, zp, zp)
        print(k, zp, "ok", flush=True)


def _grouped(dtype: str) -> None:
    from tests import test_gpu_moe as tm
    for g, zp in ((64, False), (64, True), (32, False), (32, True), (-1, False)):
        tm.test_moe_gemm_within_tolerance((1100, 3, 2, 192, 7424, g, dtype, zp, False, zp, 64, True))
        print(g, zp, "ok", flush=True)
    for wtype in ("mxfp4", "uint4b8") if dtype == "bf16" else ("uint4b8/fp16",):
        tm.test_full_size_grouped_gemm_agrees_with_dense_rows(2300, 640, 4352, wtype)
    if dtype == "bf16":
        tm.test_full_size_grouped_gemm_agrees_with_dense_rows(1100, 14336, 1024, "uint4b8")


def _oracle(dtype: str) -> None:
    from tests import gpu_util as gu
    from tests import test_gpu_parity as tp
    # 2100 rows: the last row tile has 52; 7360 columns: 192 of the last 256.  Steps of 64 rows: 3, 1, 2, 4, 7
    for m, k, n, g, zp in ((2100, 192, 7360, 64, False), (2100, 192, 7360, 64, True), (2100, 64, 7360, 32, False),
                           (2100, 128, 7360, 32, True), (2177, 256, 7424, 128, True), (2049, 448, 8192, 64, False)):
        tp.test_wide_tile_kernel_forms_within_tolerance(gu, dtype, m, k, n, g, zp, zp)
        print(m, k, n, g, zp, "ok", flush=True)
    if dtype == "bf16":
        for m, k, n in ((2100, 192, 7360), (2049, 64, 8192), (2304, 320, 7424)):
            tp.test_mxfp4_weights_dequant_bit_exact_and_gemm_within_tolerance(gu, m, k, n, True)
            print(m, k, n, "mxfp4 ok", flush=True)


def _digest(t: torch.Tensor) -> str:
    return hashlib.sha256(t.contiguous().view(torch.uint8).cpu().numpy().tobytes()).hexdigest()[:16]


def _dense() -> None:
    from sonar_amd import marlin_utils as mu, ops
    from sonar_amd.scalar_type import scalar_types
    for dtype, m, k, n, g, zp in ((torch.float16, 2100, 1152, 7360, 128, False), (torch.bfloat16, 2100, 576, 7360, 64, True),
                                  (torch.float16, 2817, 640, 8192, 32, True), (torch.bfloat16, 6400, 1024, 5056, 512, False)):
        gen = torch.Generator(device=DEV).manual_seed(m + k)
        q = torch.randint(-2 ** 31, 2 ** 31 - 1, (k // 16, 2 * n), dtype=torch.int32, device=DEV, generator=gen)
        s = (torch.rand((k // g, n), device=DEV, generator=gen) * 9e-3 + 1e-3).to(dtype)
        z = torch.randint(-2 ** 31, 2 ** 31 - 1, (k // g, n // 8), dtype=torch.int32, device=DEV, generator=gen) if zp else None
        a = torch.randn((m, k + 64), device=DEV, generator=gen).to(dtype)[:, :k]   # (rows further apart than they are long)
        empty = torch.empty(0, dtype=torch.int32, device=DEV)
        c = ops.marlin_gemm(a, None, q, None, s, None, None, z if zp else empty, empty, empty, mu.marlin_make_workspace_new(torch.device(DEV)),
                            scalar_types.uint4 if zp else scalar_types.uint4b8, m, n, k, True, False, True, False)
        assert bool(torch.isfinite(c).all())
        print(dtype, m, k, n, g, zp, _digest(c), flush=True)


def _layers() -> None:
    from sonar_amd import fused_moe
    from sonar_amd.scalar_type import scalar_types
    from tests.test_gpu_moe_gated_tiles import _experts
    # K in no more than 15 steps, so that no other kernel cuts it; one expert with most rows, one with none; ragged ends
    for kind, dtype, m, inter, k, activation, on_input in (
            ("uint4b8", torch.float16, 900, 384, 320, "silu", False), ("uint4b8", torch.bfloat16, 1500, 384, 576, "swigluoai", False),
            ("uint4", torch.float16, 900, 448, 320, "silu", True), ("uint4", torch.bfloat16, 1100, 640, 704, "silu", False),
            ("mxfp4", torch.bfloat16, 1500, 352, 320, "swigluoai", True), ("mxfp4", torch.bfloat16, 2000, 384, 128, "gelu", False)):
        e, top_k = 6, 2
        gen = torch.Generator(device=DEV).manual_seed(inter + k + m)
        w1, s1, z1 = _experts(gen, kind, e, k, 2 * inter, dtype)
        w2, s2, z2 = _experts(gen, kind, e, inter, k, dtype)
        bias1 = (torch.randn((e, 2 * inter), device=DEV, generator=gen) * 0.1).to(dtype)
        x = torch.randn((m, k), device=DEV, generator=gen).to(dtype)
        logits = torch.randn((m, e), device=DEV, generator=gen)
        logits[:, 0] += 3.0
        logits[:, 2] -= 100.0
        weights, ids = torch.topk(torch.softmax(logits, dim=1), top_k, dim=1)
        wtype = {"uint4b8": scalar_types.uint4b8, "uint4": scalar_types.uint4, "mxfp4": scalar_types.float4_e2m1f}[kind]
        out = fused_moe.fused_marlin_moe(x, w1, w2, bias1, None, s1, s2, weights.contiguous(), ids.to(torch.int32), wtype.id,
                                         activation=activation, apply_router_weight_on_input=on_input,
                                         w1_zeros=z1, w2_zeros=z2)
        assert bool(torch.isfinite(out).all())
        print(kind, dtype, m, inter, k, activation, _digest(out), flush=True)


if __name__ == "__main__":
    {"oracle": _oracle, "grouped": _grouped, "dense": _dense, "layers": _layers, "small_groups": _small_groups}[sys.argv[1]](*sys.argv[2:])
    print("done", flush=True)
