"""The digit form of the fused native GEMM (results at most 16 columns wide
whose planes x columns fill few 16-column groups): every group count, row
counts around a wave's 32 and a workgroup's 128, K around a step of 16
elements and a slice, more slices than the workspace holds weights for at
once, more rows than it holds residues for, odd K and strides, int64 and uint64
over the full range with the extremes placed. Planes against the oracle.
tests/test_dispatch.py checks on the CPU that every shape runs this form
and that the two last ones run in parts."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import oracle
import rns8_amd as r
from rns8_amd import hip, inputs

pytestmark = pytest.mark.gpu


# (m, n, k, planes, elements of a row of A past k)
SHAPES = [
    (16, 1, 1, 16, 1), (31, 1, 15, 10, 1), (33, 1, 17, 16, 1), (127, 2, 31, 10, 3), (129, 3, 255, 9, 1),
    (128, 5, 257, 9, 1), (112, 6, 511, 9, 1), (257, 4, 1040, 20, 0), (160, 7, 300, 9, 2), (140, 2, 4099, 5, 1),
    (520, 8, 520, 9, 0), (513, 9, 513, 9, 1), (300, 8, 1000, 6, 0), (144, 4, 272, 20, 0), (20000, 1, 3, 7, 1),
]
# the weights of 560000 elements in two parts of the slices; 839000 rows'
# residues of five groups in two parts of the rows
PARTS = [(16, 1, 560000, 16, 2), (839000, 4, 8, 20, 0)]


@pytest.mark.parametrize("signed", [True, False])
@pytest.mark.parametrize("m,n,k,prefix,lda_extra", SHAPES + PARTS)
def test_fused_digits_planes(gpu_ctx, signed, m, n, k, prefix, lda_extra):
    ctx = gpu_ctx
    lda, ldb = k + lda_extra, n + 1
    assert lda % 2 == 0
    dt = np.int64 if signed else np.uint64
    A = inputs.splitmix64(31 * m + k, m * lda).reshape(m, lda).view(dt)
    B = inputs.splitmix64(37 * n + k, k * ldb).reshape(k, ldb).view(dt)
    lo, hi = np.iinfo(dt).min, np.iinfo(dt).max
    A[0, 0], A[m - 1, k - 1], B[0, 0], B[k - 1, n - 1] = lo, hi, hi, lo
    sem, bk = ((r.BOUNDED_I64, r.BOUND_GLOBAL_MAX_ABS) if signed else (r.BOUNDED_U64, r.BOUND_GLOBAL_MAX_UNSIGNED))
    plan = r.Plan(ctx, r.gemm_desc(sem, bk, m, n, k, bound=1, max_prefix=prefix, flags=r.PLAN_FORCE_FIXED_PREFIX))
    C = r.Matrix(ctx, r.matrix_desc(m, n, sem, bk, prefix))
    ws = r.Workspace(ctx, plan)
    fn = r.lib().rns8_mi355x_gemm_native_i64_async if signed else r.lib().rns8_mi355x_gemm_native_u64_async
    dA, dB = hip.malloc(A.nbytes), hip.malloc(B.nbytes)
    try:
        hip.to_device(dA, A)
        hip.to_device(dB, B)
        r.check(fn(ctx.ptr, plan.ptr, ctypes.c_void_p(dA), lda, ctypes.c_void_p(dB), ldb, C.ptr, ws.ptr, None), "gemm")
        hip.synchronize()
    finally:
        hip.free(dA)
        hip.free(dB)
    pack = oracle.pack_i64 if signed else oracle.pack_u64
    want = oracle.gemm_rns(pack(np.ascontiguousarray(A[:, :k]), prefix), pack(np.ascontiguousarray(B[:, :n]), prefix),
                           prefix)
    np.testing.assert_array_equal(C.read_residues(), want)
