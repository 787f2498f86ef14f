"""The pack-time summaries of exact-wide operands at the edges of the summary
kernel's split: rows of one wave and of eight, column groups of eight,
register chunks of 512 rows and 2048 columns held and re-read, odd row
strides, row strides that need 64-bit lane offsets (2^21), long axes of either
direction that run in the tile form (ragged tiles, one and several tile
columns), and two packs into one matrix in a row (the second one's maximum must
not see the first one's). Every field against oracle/exact_range.py."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import rns8_amd as r
from oracle import exact_range as xr
from rns8_amd import hip, inputs

pytestmark = pytest.mark.gpu

FIELDS = ("max_magnitude", "absolute_sum", "sum", "minimum", "maximum", "deviation_sum")


@pytest.mark.parametrize("signed", [True, False])
@pytest.mark.parametrize(
    "rows,cols,ld",
    [(1, 1, 1), (9, 8, 8), (8, 9, 11), (513, 17, 18), (1025, 7, 7), (511, 16, 16), (2050, 3, 4), (1024, 130, 130),
     (3, 2047, 2048), (2, 2049, 2049), (17, 4100, 4100),
     (3, 70, 1 << 21), (3, 5000, 1 << 21), (8191, 3, 3), (5, 8191, 8191),
     # few axes of 8192 values and more: the tile form
     (1, 8192, 8192), (8192, 1, 1), (70, 8200, 8203), (8257, 65, 66), (2, 65700, 65700)],
)
def test_axes_edges(gpu_ctx, signed, rows, cols, ld):
    ctx = gpu_ctx
    sem = r.EXACT_WIDE_SIGNED if signed else r.EXACT_WIDE_UNSIGNED
    M = r.Matrix(ctx, r.matrix_desc(rows, cols, sem, r.BOUND_NONE, 20))
    pack = r.lib().rns8_mi355x_pack_i64_device if signed else r.lib().rns8_mi355x_pack_u64_device
    for turn in range(2):
        x = inputs.splitmix64(77 * rows + cols + turn, rows * cols).reshape(rows, cols)
        if turn:  # a smaller range than the first pack's
            x = x >> np.uint64(3)
        elif rows * cols > 1:
            x[0, 0] = np.uint64(1 << 63)
            x[-1, -1] = np.uint64((1 << 63) - 1)
        if signed:
            x = x.view(np.int64)
        staged = np.full((rows, ld), -1 if signed else 0xFFFFFFFFFFFFFFFF, dtype=x.dtype)
        staged[:, :cols] = x  # padding is not part of the operand
        d = hip.malloc(staged.nbytes)
        try:
            hip.to_device(d, staged)
            r.check(pack(ctx.ptr, M.ptr, ctypes.c_void_p(d), ld, 0, None), "pack")
            hip.synchronize()
        finally:
            hip.free(d)
        bound, kind, got_rows, got_cols = M.exact_proof(ctx)
        want = xr.native_operand([[int(v) for v in row] for row in x])
        assert kind == r.EXACT_AXES_NATIVE and bound == want.max_magnitude
        for got, axes in ((got_rows, want.rows), (got_cols, want.cols)):
            assert len(got) == len(axes)
            for i, (g, w) in enumerate(zip(got, axes)):
                assert all(g[f] == getattr(w, f) for f in FIELDS), (turn, i, g)


def test_pack_after_overlapping_packs(gpu_ctx):
    """Packs of one matrix on two streams at once are a caller's error and may
    spoil their own proofs, but not the next pack's: with an ordered pack
    behind them, of smaller values, the matrix's maximum and summaries are that
    pack's."""
    ctx = gpu_ctx
    rows, cols = 6000, 40
    pack = r.lib().rns8_mi355x_pack_i64_device
    M = r.Matrix(ctx, r.matrix_desc(rows, cols, r.EXACT_WIDE_SIGNED, r.BOUND_NONE, 20))
    big = inputs.splitmix64(91, rows * cols).reshape(rows, cols).view(np.int64)
    small = big >> np.int64(40)
    d_big, d_small = hip.malloc(big.nbytes), hip.malloc(small.nbytes)
    streams = [hip.stream_create(), hip.stream_create()]
    try:
        hip.to_device(d_big, big)
        hip.to_device(d_small, small)
        for turn in range(4):
            for _ in range(20):
                for s in streams:
                    r.check(pack(ctx.ptr, M.ptr, ctypes.c_void_p(d_big), cols, 0, ctypes.c_void_p(s)), "pack")
            hip.synchronize()
            r.check(pack(ctx.ptr, M.ptr, ctypes.c_void_p(d_small), cols, 0, None), "pack")
            hip.synchronize()
            bound, kind, got_rows, got_cols = M.exact_proof(ctx)
            assert kind == r.EXACT_AXES_NATIVE and bound == int(np.abs(small).max()), turn
            for axis, got in ((1, got_rows), (0, got_cols)):
                want = small.sum(axis=axis)
                assert [g["sum"] for g in got] == [int(v) for v in want], turn
    finally:
        hip.synchronize()
        for s in streams:
            hip.stream_destroy(s)
        hip.free(d_big)
        hip.free(d_small)
