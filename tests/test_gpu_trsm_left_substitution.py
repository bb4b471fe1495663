"""Left-side triangular solves above 64 rows are substitutions: backward stable
whatever the condition of the triangle's blocks, and an Inf or NaN reaches only
the rows that depend on it (as in driver/level3/trsm_L.c with
kernel/generic/trsm_kernel_LT.c).

Residual bound, per element, for op(A) X = B solved row by row with one rounding
per term and a reciprocal diagonal (3 roundings per division), sums in any
order: |op(A) X - B| <= (m + 3) eps (|op(A)||X| + |B|) to first order; 2 m eps
is allowed (m >= 65).
"""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

FORMS = [(lo, tr, un) for lo in (0, 1) for tr in (0, 1) for un in (0, 1)]


def solve(oba, dt, lower, trans, unit, A, B):
    """X of op(A) X = B (Fortran-ordered host arrays); A's other triangle goes in as NaN."""
    L = oba.lib()
    f = L.cblas_dtrsm if dt == np.float64 else L.cblas_strsm
    m, n = B.shape
    keep = np.tril(np.ones((m, m), bool)) if lower else np.triu(np.ones((m, m), bool))
    dA = oba.DeviceBuffer.from_array(np.asfortranarray(np.where(keep, A, np.nan).astype(dt)))
    dB = oba.DeviceBuffer.from_array(np.asfortranarray(B.astype(dt)))
    f(102, 141, 122 if lower else 121, 112 if trans else 111, 132 if unit else 131, m, n, 1.0, dA.ptr, m, dB.ptr, m)
    return dB.to_array(np.empty((m, n), dt, order="F"))


def triangle(rng, kind, m, lower, unit, dt):
    if kind == "minus_ones":
        T = -np.ones((m, m))
        d = np.ones(m)
    elif kind == "uniform":
        T = rng.uniform(-1, 1, (m, m))
        d = rng.uniform(0.5, 1, m)
    elif kind == "positive":
        T = rng.uniform(0, 1, (m, m)) * (0.5 if m > 128 else 1.0)
        d = rng.uniform(0.5, 1, m)
    else:
        T = rng.standard_normal((m, m)) * (0.5 if m > 128 else 1.0)
        d = rng.uniform(0.5, 2, m)
    T = np.tril(T, -1) if lower else np.triu(T, 1)
    return (T + np.diag(np.ones(m) if unit else d)).astype(dt)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("m", [65, 128, 256, 300])
@pytest.mark.parametrize("kind", ["minus_ones", "uniform", "positive", "normal"])
def test_backward_error(oba, dt, m, kind):
    rng = np.random.default_rng(m)
    eps = np.finfo(dt).eps
    n = 17
    for lower, trans, unit in FORMS:
        A = triangle(rng, kind, m, lower, unit, dt)
        M = (A.T if trans else A).astype(np.longdouble)
        x = rng.integers(-4, 5, (m, n)).astype(dt)
        B = (M @ x).astype(dt)
        X = solve(oba, dt, lower, trans, unit, A, B)
        R = np.abs(M @ X - B)
        bound = 2 * m * eps * (np.abs(M) @ np.abs(X) + np.abs(B))
        assert np.isfinite(X).all(), (lower, trans, unit)
        assert np.all(R <= bound), (lower, trans, unit, float((R / np.maximum(bound, 1e-300)).max()))
        if kind == "minus_ones":   # integers throughout
            assert np.array_equal(X, x), (lower, trans, unit)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("m", [65, 130, 256, 300])
def test_nonfinite_reaches_dependent_rows_only(oba, dt, m):
    rng = np.random.default_rng(m)
    rows = sorted({0, 15, 16, 40, 63, 64, m // 2, m - 2, m - 1})
    n = 2 * len(rows)
    for lower, trans, unit in FORMS:
        A = triangle(rng, "uniform", m, lower, unit, dt)
        A = np.where(np.eye(m, dtype=bool), A, A * dt(0.125)).astype(dt)
        B = rng.standard_normal((m, n)).astype(dt)
        for i, r in enumerate(rows):   # one value of B
            B[r, 2 * i] = np.inf
            B[r, 2 * i + 1] = np.nan
        X = solve(oba, dt, lower, trans, unit, A, B)
        want = oracle.trsm(0, lower, trans, 1 - unit, 1.0, A, B)
        assert np.array_equal(np.isfinite(X), np.isfinite(want)), (lower, trans, unit)
        for r, c in ((m - 1, m - 20), (40, 3), (m // 2, m // 2 - 1)):   # one value of the triangle
            A2 = A.copy()
            A2[(r, c) if lower else (c, r)] = np.nan
            B2 = rng.standard_normal((m, 3)).astype(dt)
            X = solve(oba, dt, lower, trans, unit, A2, B2)
            want = oracle.trsm(0, lower, trans, 1 - unit, 1.0, A2, B2)
            assert np.array_equal(np.isfinite(X), np.isfinite(want)), (lower, trans, unit, r, c)


def test_gesv_many_right_hand_sides(oba):
    """A = L U with U's blocks near overflow of an inverse: more than 16
    right-hand sides keep the backward error of few."""
    L = oba.lib()
    rng = np.random.default_rng(3)
    n = 130
    U = np.triu(rng.uniform(-1, 1, (n, n)), 1) + np.diag(np.ones(n))
    Lo = np.tril(rng.uniform(-1, 1, (n, n)), -1) / 4 + np.eye(n)
    A = Lo @ U
    for nrhs in (3, 17, 40):
        B = rng.standard_normal((n, nrhs))
        dA, dB = oba.DeviceBuffer.from_array(np.asfortranarray(A)), oba.DeviceBuffer.from_array(np.asfortranarray(B))
        piv = oba.DeviceBuffer(4 * n)
        info = ctypes.c_int(-1)
        L.dgesv_(oba.ip(n), oba.ip(nrhs), dA.ptr, oba.ip(n), piv.ptr, dB.ptr, oba.ip(n), ctypes.byref(info))
        X = dB.to_array(np.empty((n, nrhs), order="F"))
        F = dA.to_array(np.empty((n, n), order="F"))
        assert info.value == 0
        Lf, Uf = np.tril(F, -1) + np.eye(n), np.triu(F)
        R = np.abs(A.astype(np.longdouble) @ X - B)
        bound = 4 * n * np.finfo(np.float64).eps * (np.abs(Lf) @ (np.abs(Uf) @ np.abs(X))).max(axis=0)
        assert np.all(R.max(axis=0) <= bound), float((R.max(axis=0) / bound).max())
