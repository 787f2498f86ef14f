"""Every output tile of the plane GEMM (256x256, 256x128, 128x256, 128x128,
64x64) at its edges: rows and columns one past and one short of a tile, K of
one element, around the 64-deep step and the 128-deep A chunk, odd chunk
counts, several tiles of one chunk per workgroup, and tile counts that leave some workgroups of the grid without a tile. Finite products, compared with float64 matrix products on the CPU
(k * 255^2 < 2^53: every sum is exact)."""
from __future__ import annotations

import numpy as np
import pytest

import rns8_amd as r
from rns8_amd import inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "tile,m,n,k",
    [
        ("64x64", 1, 17, 1), ("64x64", 63, 65, 63), ("64x64", 65, 64, 65), ("64x64", 130, 127, 127),
        ("64x64", 64, 191, 129), ("64x64", 200, 300, 1000), ("64x64", 190, 180, 70), ("64x64", 97, 338, 1058),
        ("128x128", 2049, 1030, 260), ("128x128", 2050, 1025, 385), ("128x128", 2709, 707, 20),
        ("128x128", 4200, 4300, 100), ("128x128", 4200, 4300, 1),
        ("256x128", 1100, 4097, 1025), ("256x128", 1568, 2477, 1060),
        ("128x256", 2373, 3211, 1036),
        ("256x256", 4097, 3000, 129), ("256x256", 3439, 3594, 20), ("256x256", 4095, 4090, 641), ("256x256", 4300, 3800, 200), ("256x256", 5000, 9000, 65),
    ],
)
@pytest.mark.parametrize("modulus", [251, 256])
def test_gemm_tile_edges(gpu_ctx, tile, m, n, k, modulus):
    sem = r.FINITE_RING_U8
    desc = r.gemm_desc(sem, r.BOUND_NONE, m, n, k, finite_modulus=modulus)
    plan = r.Plan(gpu_ctx, desc)
    assert f"{tile} tile" in plan.selected_kernel()
    mats = [r.Matrix(gpu_ctx, r.matrix_desc(a, b, sem, r.BOUND_NONE)) for a, b in ((m, k), (k, n), (m, n))]
    ws = r.Workspace(gpu_ctx, plan)
    A = inputs.bytes_below(11 * m + k, (m, k), modulus)
    B = inputs.bytes_below(13 * n + k, (k, n), modulus)
    r.check(r.pack_finite_u8(gpu_ctx, mats[0], modulus, A, 1), "pack A")
    r.check(r.pack_finite_u8(gpu_ctx, mats[1], modulus, B, 2), "pack B")
    r.check(r.gemm_finite_u8(gpu_ctx, plan, modulus, *mats, ws), "gemm")
    out = np.zeros((m, n), dtype=np.uint8)
    r.check(r.export_finite_u8(gpu_ctx, plan, modulus, mats[2], out), "export")
    want = np.mod(A.astype(np.float64) @ B.astype(np.float64), modulus).astype(np.uint8)
    np.testing.assert_array_equal(out, want)
