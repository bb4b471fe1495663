"""Batched LU at the edges of its size classes (64, 128, 256, 512 rows), of its
32-column panels, 8-column blocks and 16-row tiles, square, tall and wide, with
padded leading dimensions: a valid partial-pivoting factorization (backward
error, |l| <= 1), FP64 pivots and info as the oracle's, padding untouched, and
the pivot rules for zero, subnormal and NaN columns.

Tolerance: the computed factors satisfy P A + E = L U with
|E| <= gamma_k |L| |U|, gamma_k ~ k*eps (k = min(m, n)); one more rounding per
element for the stored reciprocal makes the factor 2.
"""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _run(oba, dt, mats, ldas):
    L = oba.lib()
    f = L.openblas_amd_dgetrf_batch if dt == np.float64 else L.openblas_amd_sgetrf_batch
    bufs, pivs = [], []
    for a, ld in zip(mats, ldas):
        b = np.full((ld, a.shape[1]), 7.5, dt, order="F")
        b[:a.shape[0]] = a
        bufs.append(b)
        pivs.append(np.full(max(min(a.shape), 1), -5, np.int32))
    cnt = len(mats)
    info = np.full(cnt, -99, np.int32)
    ia = lambda v: (ctypes.c_int * len(v))(*v)
    pa = lambda v: (ctypes.c_void_p * len(v))(*v)
    r = f(ia([a.shape[0] for a in mats]), ia([a.shape[1] for a in mats]), pa([b.ctypes.data for b in bufs]), ia(ldas),
          pa([p.ctypes.data for p in pivs]), info.ctypes.data_as(ctypes.POINTER(ctypes.c_int)), cnt)
    assert r == 0
    return bufs, pivs, info


def _check(dt, a, b, piv, info, same):
    m, n = a.shape
    k = min(m, n)
    lu = b[:m]
    assert np.all(b[m:] == 7.5)
    luo, pivo, infoo = oracle.getf2(a)
    assert info == infoo
    if same:
        assert np.array_equal(piv[:k], pivo)
    lm = (np.tril(lu, -1)[:, :k] + np.eye(m, k)).astype(np.float64)
    um = np.triu(lu)[:k].astype(np.float64)
    assert np.abs(lm).max(initial=0) <= 1.0
    pa = oracle.laswp(a.astype(np.float64), 1, k, piv[:k], 1)
    e = np.abs(lm @ um - pa)
    assert np.all(e <= 2 * (k + 1) * np.finfo(dt).eps * (np.abs(lm) @ np.abs(um)) + np.finfo(dt).tiny)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("rows", [(1, 7, 8, 9, 15, 16, 17, 31, 32, 33), (63, 64, 65, 96, 97), (127, 128, 129, 160),
                                  (255, 256, 257), (480, 511, 512)])
def test_getrf_batch_edges(oba, dt, rows):
    rng = np.random.default_rng(rows[0] + (dt == np.float32))
    mats, ldas = [], []
    for m in rows:
        for n in {1, 31, 33, m, max(1, m - 1), m + 1, m + 130}:
            mats.append(rng.standard_normal((m, n)).astype(dt))
            ldas.append(m + int(rng.integers(0, 4)))
    for a, b, p, i in zip(mats, *_run(oba, dt, mats, ldas)):
        _check(dt, a, b, p, i, dt == np.float64)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_getrf_batch_special_columns(oba, dt):
    rng = np.random.default_rng(5)
    mats = []
    for n in (20, 64, 100, 130, 300):
        a = rng.integers(-1, 2, (n, n)).astype(dt)          # ties in every early column
        mats.append(a + 4 * np.eye(n, dtype=dt)[rng.permutation(n)])
        z = rng.standard_normal((n, n)).astype(dt)
        z[:, n // 2] = 0                                    # exact zero column: info
        mats.append(z)
    for a, b, p, i in zip(mats, *_run(oba, dt, mats, [a.shape[0] for a in mats])):
        _check(dt, a, b, p, i, False)
    # the first column decides by itself: ties to the lowest row, a NaN only at
    # its own position, a subnormal pivot neither scales nor is an error
    one = []
    for n, where in ((40, 0), (40, 30), (70, 69), (200, 150)):
        c = np.full((n, 1), -2.0, dt)
        one.append(c.copy())                                # all equal: row 1
        c[where] = np.nan
        one.append(c.copy())                                # NaN
        c[:] = 0
        c[where] = np.finfo(dt).tiny / 4
        one.append(c.copy())                                # subnormal
    for a, b, p, i in zip(one, *_run(oba, dt, one, [a.shape[0] for a in one])):
        luo, pivo, infoo = oracle.getf2(a)
        assert i == infoo and np.array_equal(p, pivo), (a.shape, p, pivo)
        if np.nanmax(np.abs(a)) < np.finfo(dt).tiny:        # interchanged, not scaled
            luo = oracle.laswp(a, 1, 1, p, 1)
        assert np.array_equal(b, luo, equal_nan=True)
