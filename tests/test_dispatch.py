"""Dispatch rules asked of the library's own objects (CPU), through
tests/dispatch_check.cpp: which form of the fused native GEMM a product runs
(fused.hip, fused_skinny.hip, fused_digits.hpp; the digit form is expected where
it measured faster and the residue form where that did), and the plane GEMM's
persistent grid."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

import test_gpu_fused_digits as digits
import test_gpu_fused_skinny as skinny

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "rns8_amd" / "csrc"
OBJS = [ROOT / "rns8_amd" / "_build" / f"{p.stem}.o" for p in sorted([*CSRC.glob("*.hip"), *CSRC.glob("*.cpp")])]


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    if not all(p.is_file() for p in OBJS):
        pytest.skip("library objects missing: run __graft_entry__.build()")
    exe = tmp_path_factory.mktemp("dispatch") / "dispatch_check"
    subprocess.run([gxx, "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include", "-I",
                    str(CSRC), "-I", str(ROOT / "include"), str(ROOT / "tests" / "dispatch_check.cpp"),
                    *map(str, OBJS), "-L/opt/rocm/lib", "-Wl,-rpath,/opt/rocm/lib", "-lamdhip64", "-pthread", "-o",
                    str(exe)], check=True)

    def run(what, cases):
        text = "\n".join(" ".join([what, *map(str, c)]) for c in cases) + "\n"
        res = subprocess.run([str(exe)], input=text, capture_output=True, text=True, timeout=60, check=True)
        return [line.split() for line in res.stdout.splitlines()]

    return run


@pytest.fixture(scope="module")
def forms(ask):
    return lambda shapes: ask("fused", shapes)


# (m, n, k, planes)
RESIDUE_FASTER = [
    # small products, bound by their launches
    (16, 1, 8, 9), (16, 1, 100, 7), (1000, 1, 64, 7), (1000, 2, 100, 8), (128, 1, 100, 7), (4096, 4, 128, 9),
    # deep ones of few rows, where writing the weights costs more than the residues
    (128, 7, 200000, 9), (128, 4, 65536, 9), (800, 7, 32768, 9), (16, 1, 560000, 7), (952, 6, 103079, 7),
    (52, 6, 130359, 5), (115, 5, 440956, 7), (64, 2, 560000, 9), (200, 7, 65536, 9),
    # five and six planes
    (1160, 10, 6968, 6), (5748, 5, 6620, 5), (53, 5, 53387, 6),
    # many groups for the planes
    (8192, 8, 8192, 9), (200, 16, 3000, 18), (8, 8, 1 << 20, 9),
]
DIGITS_FASTER = [
    (8192, 1, 8192, 9), (8192, 7, 8192, 9), (2000, 7, 1000, 9), (128, 7, 256, 9), (200, 4, 20000, 20), (512, 3, 512, 5),
    (2000, 9, 1000, 9), (64, 2, 8000, 9), (16, 1, 100000, 9), (30000, 1, 64, 7), (200000, 1, 8, 9), (128, 3, 200, 8),
    (1200, 4, 65536, 9), (512, 2, 100000, 9), (200, 4, 65536, 20), (16, 1, 560000, 16), (5041, 7, 1192, 6),
]


def test_forms_taken_are_the_faster_ones(forms):
    got = [f[0] for f in forms(RESIDUE_FASTER)]
    assert got == ["residue"] * len(RESIDUE_FASTER), [s for s, g in zip(RESIDUE_FASTER, got) if g != "residue"]
    got = [f[0] for f in forms(DIGITS_FASTER)]
    assert got == ["digits"] * len(DIGITS_FASTER), [s for s, g in zip(DIGITS_FASTER, got) if g != "digits"]


def test_gpu_tests_run_the_forms_they_are_for(forms):
    assert [f[0] for f in forms([s[:4] for s in digits.SHAPES + digits.PARTS])] == ["digits"] * len(
        digits.SHAPES + digits.PARTS)
    assert [f[0] for f in forms([c[:4] for c in skinny.CASES])] == skinny.FORMS
    assert [f[0] for f in forms([e[:4] for e in skinny.EXTENTS])] == [e[4] for e in skinny.EXTENTS]


def test_gpu_test_shapes_run_in_parts(forms):
    """The workspace holds at most 64 MiB of weights and of residues at once
    (plus one slice's, one row group's, rounding): these products have more of
    either, so they run in parts of it."""
    limit = 64 << 20
    (wm, wn, wk, wp, _), (rm, rn, rk, rp, _) = digits.PARTS
    (_, w_slices, w_ks, w_bytes), (_, r_slices, _, r_bytes) = forms([digits.PARTS[0][:4], digits.PARTS[1][:4]])
    groups = -(-wn * wp // 16)
    all_weights = int(w_slices) * int(w_ks) // 16 * 2048 * groups
    residues = int(w_slices) * 16 * groups * wm
    assert all_weights > limit and int(w_bytes) < all_weights + residues
    groups = -(-rn * rp // 16)
    all_residues = int(r_slices) * 16 * groups * rm
    assert all_residues > limit and int(r_bytes) < all_residues


@pytest.mark.parametrize("slots", [256, 512, 1024])
def test_persistent_grid_runs_every_unit_once(ask, slots):
    """The plane GEMM's unit walk (gemm.hip: XCD x owns units [x units / 8, (x +
    1) units / 8), its workgroups in lock step; grids that are no multiple of 8
    walk all units) reaches every unit once, and no workgroup has a second unit
    while a slot is free."""
    counts = [*range(1, slots + 40), 3 * slots - 1, 3 * slots, 3 * slots + 9]
    for units, (grid,) in zip(counts, ask("grid", [(u, slots) for u in counts])):
        grid = int(grid)
        assert 0 < grid <= slots
        seen, most = [], 0
        for b in range(grid):
            if grid % 8 == 0:
                x = b & 7
                mine = list(range(x * units // 8 + (b >> 3), (x + 1) * units // 8, grid >> 3))
            else:
                mine = list(range(b, units, grid))
            seen += mine
            most = max(most, len(mine))
        assert sorted(seen) == list(range(units)), units
        assert most == -(-units // slots), (units, grid)
