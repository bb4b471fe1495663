"""FP64 GEMM on 128x128 tiles (at least 8 tiles per CU and K >= 4096), odd sizes,
all four forms: C x against A (B x) for three vectors of +-1.  Each entry of C
is within (k+2)*eps*|A||B| of the exact one and the two sides' products add
(n+k+2)*eps of the same, so (n+2k+4)*eps*|A|(|B||x|) bounds the difference.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_dgemm_large_tiles(oba, ta, tb):
    m, n, k = 5795, 5801, 4099
    rng = np.random.default_rng(1 + ta + 2 * tb)
    a = rng.uniform(-1, 1, (m, k) if ta else (k, m))   # rows are columns of the operand
    b = rng.uniform(-1, 1, (k, n) if tb else (n, k))
    c = np.full((n, m + 1), np.nan)
    da, db, dc = (oba.DeviceBuffer.from_array(v) for v in (a, b, c))
    oba.lib().cblas_dgemm(102, 112 if ta else 111, 112 if tb else 111, m, n, k, 0.5, da.ptr, k if ta else m, db.ptr,
                          n if tb else k, 0.0, dc.ptr, m + 1)
    c = dc.to_array(c)
    assert np.isnan(c[:, m]).all()
    A, B = (a if ta else a.T), (b if tb else b.T)
    x = rng.integers(0, 2, (n, 3)) * 2.0 - 1.0
    got, want = c[:, :m].T @ x, 0.5 * (A @ (B @ x))
    bound = (n + 2 * k + 4) * np.finfo(np.float64).eps * 0.5 * (np.abs(A) @ (np.abs(B) @ np.abs(x)))
    assert np.all(np.abs(got - want) <= bound)
