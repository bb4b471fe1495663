"""The FP32 form of the LU leaf panel (its records hold two elements a word, an
odd one at the end, and position and reciprocal in one) at the edges of its
workgroups and widths.  Random data: a valid partial-pivoting factorization with
a dget01 ratio below 30.  Pivots and INFO equal to the oracle's where FP32 is
exact: the columns with a choice hold small powers of two, the other columns one
entry each, and no row has entries in two columns, so nothing is rounded."""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

SIZES = [(31, 31), (64, 33), (511, 32), (512, 40), (513, 31), (513, 64), (1025, 65), (1537, 96), (4000, 32), (16384, 34),
         (16385, 34)]


def run(oba, A):
    m, n = A.shape
    F = np.array(A, np.float32, order="F")
    piv = np.zeros(min(m, n), np.int32)
    info = ctypes.c_int(-1)
    oba.lib().sgetrf_(oba.ip(m), oba.ip(n), F.ctypes.data, oba.ip(m), piv.ctypes.data, ctypes.byref(info))
    return F, piv, info.value


@pytest.mark.parametrize("m,n", SIZES)
def test_random(oba, m, n):
    A = np.random.default_rng(m + n).standard_normal((m, n)).astype(np.float32)
    F, piv, info = run(oba, A)
    k = min(m, n)
    assert info == 0 and np.all(piv >= np.arange(1, k + 1)) and np.all(piv <= m)
    L = np.tril(F[:, :k], -1).astype(np.float64)
    assert np.abs(L).max() <= 1
    L[np.arange(k), np.arange(k)] = 1
    P = oracle.laswp(A.astype(np.float64), 1, k, piv, 1)
    R = np.abs(P - L @ np.triu(F[:k]).astype(np.float64))
    assert R.sum(0).max() / (np.abs(A).sum(0).max() * n * np.finfo(np.float32).eps) < 30


def exact_matrix(rng, m, n, choice):
    """columns in `choice` of powers of two with several largest entries, the others of one entry; no row in two columns"""
    A = np.zeros((m, n), np.float32)
    rows = rng.permutation(m)
    single = [c for c in range(min(m, n)) if c not in choice]
    own = rows[:len(single)]
    A[own, single] = 2.0 ** rng.integers(-3, 4, len(single)) * rng.choice([-1, 1], len(single))
    rest = rng.permutation(np.setdiff1d(np.arange(m), own))
    for c, r in zip(sorted(choice), np.array_split(rest, len(choice))):   # rows of their own, too
        A[r, c] = rng.choice([0, 0.5, 1, 2, 2], len(r)) * rng.choice([-1, 1], len(r))
    return A


@pytest.mark.parametrize("m,n", SIZES)
@pytest.mark.parametrize("kind", ["ties", "zeros"])
def test_exact_pivots(oba, m, n, kind):
    rng = np.random.default_rng(3 * m + n)
    k = min(m, n)
    if kind == "ties":
        A = exact_matrix(rng, m, n, {0, k // 2, k - 1})
    else:
        A = exact_matrix(rng, m, n, {1})
        A[:, [0, k // 2]] = 0
    F, piv, info = run(oba, A)
    oF, opiv, oinfo = oracle.getf2(A)
    assert info == oinfo and np.array_equal(piv, opiv)
    assert np.array_equal(F, oF)


@pytest.mark.parametrize("m", [300, 1300])
@pytest.mark.parametrize("at", [0, 7])
@pytest.mark.parametrize("what", [np.nan, np.inf])
def test_nonfinite(oba, m, at, what):
    rng = np.random.default_rng(m + at)
    for where in ("pivot position", "elsewhere"):
        A = exact_matrix(rng, m, 40, {at})
        order = oracle.getf2(A)[1][:at]
        rows = np.arange(m)
        for j, p in enumerate(order):
            rows[[j, p - 1]] = rows[[p - 1, j]]
        A[rows[at] if where == "pivot position" else rows[-1], at] = what   # the row that is at position `at` then
        F, piv, info = run(oba, A)
        oF, opiv, oinfo = oracle.getf2(A)
        assert info == oinfo and np.array_equal(piv[:at + 1], opiv[:at + 1]), where
        assert np.array_equal(np.isfinite(F[:, :at + 1]), np.isfinite(oF[:, :at + 1])), where


@pytest.mark.parametrize("m", [300, 1300])
def test_row_of_all_bits(oba, m):
    """a pivot row whose words are all ones, which is what an empty record holds"""
    A = np.random.default_rng(m).standard_normal((m, 33)).astype(np.float32)
    A[0] = np.full(33, 0xFFFFFFFF, np.uint32).view(np.float32)
    F, piv, info = run(oba, A)
    assert piv[0] == 1 and info == 0 and np.isnan(F[0]).all() and np.isnan(F[1:, 1:]).all()
