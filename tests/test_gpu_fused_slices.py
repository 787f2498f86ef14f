"""The tile form of the fused native GEMM: odd plane counts (the last workgroup
of planes holds one), tiles cut by rows and columns, and inner dimensions whose
slices fill one to three rounds of CUs with ragged last slices. Planes against
the oracle."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import oracle
import rns8_amd as r
from rns8_amd import hip, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("signed", [True, False])
@pytest.mark.parametrize(
    "m,n,k,prefix",
    [(33, 40, 1, 1), (40, 20, 513, 3), (129, 127, 1025, 5), (17, 130, 9001, 9), (128, 17, 20000, 7), (200, 300, 3000, 9),
     (260, 64, 4097, 2), (64, 200, 12000, 5)],
)
def test_fused_tile_form_planes(gpu_ctx, signed, m, n, k, prefix):
    ctx = gpu_ctx
    lda, ldb = k + k % 2, n + n % 2 + 2
    dt = np.int64 if signed else np.uint64
    A = inputs.splitmix64(41 * m + k, m * lda).reshape(m, lda).view(dt)
    B = inputs.splitmix64(43 * n + k, k * ldb).reshape(k, ldb).view(dt)
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
