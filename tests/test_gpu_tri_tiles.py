"""The triangle-restricted GEMM's tile order (groups of 8 tile rows of the
triangle) and the 64x64 Cholesky leaves at their edges: SYRK for tile counts
around a group with NaN in the other triangle, which stays as it is, and potrf
around the 16-column steps of a leaf with a failing diagonal in each of them.
SYRK within 16 eps (|A||A|^T + |C|) per element; potrf against the oracle's
potf2 within 8 n eps of the largest entry (well-conditioned matrices), INFO and
the stored failing diagonal's sign equal, a NaN passing through.
"""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("n,k", [(31, 5), (65, 70), (250, 33), (257, 300), (511, 20), (513, 20), (577, 130), (1100, 17),
                                 (1600, 40), (2400, 9)])
@pytest.mark.parametrize("uplo", [121, 122])
def test_syrk_tiles(oba, dt, n, k, uplo):
    L = oba.lib()
    rng = np.random.default_rng(n + k)
    A = rng.uniform(-1, 1, (n, k)).astype(dt)
    C0 = rng.uniform(-1, 1, (n, n)).astype(dt)
    mine = np.triu(np.ones((n, n), bool)) if uplo == 121 else np.tril(np.ones((n, n), bool))
    C0[~mine] = np.nan
    Af, C = np.asfortranarray(A), np.asfortranarray(C0)
    f = L.cblas_dsyrk if dt == np.float64 else L.cblas_ssyrk
    f(102, uplo, 111, n, k, -1.0, Af.ctypes.data, n, 1.0, C.ctypes.data, n)
    a = A.astype(np.float64)
    ref, g = np.nan_to_num(C0).astype(np.float64) - a @ a.T, np.abs(a) @ np.abs(a).T + np.abs(np.nan_to_num(C0))
    err = np.abs(C.astype(np.float64) - ref)
    assert np.all(err[mine] <= 16 * np.finfo(dt).eps * g[mine])
    assert np.isnan(C[~mine]).all()


def potrf(oba, A, uplo):
    F = np.array(A, order="F")
    n, info = A.shape[0], ctypes.c_int(-1)
    f = oba.lib().dpotrf_ if A.dtype == np.float64 else oba.lib().spotrf_
    f(uplo, oba.ip(n), F.ctypes.data, oba.ip(n), ctypes.byref(info))
    return F, info.value


def spd(n, dt, seed):
    z = np.random.default_rng(seed).standard_normal((n, 2 * n))
    return (z @ z.T / (2 * n) + 0.1 * np.eye(n)).astype(dt)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 33, 48, 63, 64, 65, 130, 200])
@pytest.mark.parametrize("uplo", [b"L", b"U"])
def test_potrf_leaf(oba, dt, n, uplo):
    A = spd(n, dt, n)
    part = np.tril if uplo == b"L" else np.triu
    F, info = potrf(oba, A, uplo)
    ref = np.linalg.cholesky(A.astype(np.float64))
    ref = ref if uplo == b"L" else ref.T
    assert info == 0
    assert np.abs(part(F) - ref).max() <= 8 * n * np.finfo(dt).eps * np.abs(ref).max()
    assert np.array_equal(F - part(F), A - part(A))          # the other triangle
    for f in sorted({0, n // 3, n // 2, (3 * n) // 4, n - 1}):
        B = A.copy()
        B[f, f] = -1
        F, info = potrf(oba, B, uplo)
        assert info == f + 1
        got = part(F) if uplo == b"L" else part(F).T
        rl = ref if uplo == b"L" else ref.T
        # the leading part is final (rows below the failing block are not solved any more)
        assert np.abs(got[:f, :f] - rl[:f, :f]).max(initial=0) <= 8 * n * np.finfo(dt).eps * np.abs(ref).max()
        assert F[f, f] <= -1                                   # the updated diagonal, as it is
    B = A.copy()
    B[n // 2, n // 2] = np.nan                                 # not caught (ajj <= 0 is false)
    F, info = potrf(oba, B, uplo)
    assert info == 0 and np.isnan(F[n // 2, n // 2])
