"""The LU leaf panel at its edges: row counts around the workgroup (512 rows)
and around the limit of 32 workgroups, widths around the 32-column leaf and the
two-leaf node, pivots tied between workgroups (duplicate rows), zero columns,
and NaN / infinity away from and at the pivot position.  IPIV and INFO must
equal the oracle's getf2 (IAMAX's first maximum and NaN rule); the factors are
within c*n*eps of the matrix (dget01 ratio below 30).
"""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def run(oba, A):
    m, n = A.shape
    F = np.array(A, order="F")
    piv = np.zeros(min(m, n), np.int32)
    info = ctypes.c_int(-1)
    oba.lib().dgetrf_(oba.ip(m), oba.ip(n), F.ctypes.data, oba.ip(m), piv.ctypes.data, ctypes.byref(info))
    return F, piv, info.value


def dget01(A, F, piv):
    m, n = A.shape
    k = min(m, n)
    P = A.copy()
    for i, p in enumerate(piv):
        P[[i, p - 1]] = P[[p - 1, i]]
    L = np.tril(F[:, :k], -1)
    L[np.arange(k), np.arange(k)] = 1
    return np.abs(P - L @ np.triu(F[:k])).sum(0).max() / (np.abs(A).sum(0).max() * n * np.finfo(float).eps)


@pytest.mark.parametrize("m,n", [(31, 31), (64, 33), (511, 32), (512, 40), (513, 31), (513, 64), (1025, 65), (1537, 96),
                                 (4000, 32), (16384, 34), (16385, 34)])
@pytest.mark.parametrize("kind", ["random", "ties", "zeros"])
def test_panel_pivots(oba, m, n, kind):
    rng = np.random.default_rng(m + n)
    A = rng.standard_normal((m, n))
    if kind == "ties":      # the same rows again in other workgroups, in another order, some negated
        d = min(m, max(n + 3, 100))
        idx = rng.integers(0, d, m)
        idx[:d] = rng.permutation(d)
        A = A[:d][idx] * rng.choice([-1.0, 1.0], (m, 1))
    if kind == "zeros":     # exact zero columns: no interchange, INFO is the first
        A[:, [0, n // 2]] = 0
    F, piv, info = run(oba, A)
    _, opiv, oinfo = oracle.getf2(A)
    assert info == oinfo and np.array_equal(piv, opiv)
    assert dget01(A, F, piv) < 30


@pytest.mark.parametrize("m", [300, 1300])
@pytest.mark.parametrize("where", [(0, 0), (700, 0), (5, 3), (299, 1)])
@pytest.mark.parametrize("what", [np.nan, np.inf])
def test_panel_nonfinite(oba, m, where, what):
    A = np.random.default_rng(m).standard_normal((m, 40))
    A[where[0] % m, where[1]] = what
    F, piv, info = run(oba, A)
    oF, opiv, oinfo = oracle.getf2(A)
    assert info == oinfo
    # up to the column where the non-finite value enters, and that column
    assert np.array_equal(piv[:where[1] + 1], opiv[:where[1] + 1])
    assert np.array_equal(np.isfinite(F[:, :where[1] + 1]), np.isfinite(oF[:, :where[1] + 1]))
