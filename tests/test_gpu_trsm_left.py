"""Left-side triangular solves around the 64-row blocks and the 256-row leaves,
with column counts around the 16- and 32-vector workgroups, every uplo /
transpose / diagonal form, odd leading dimensions, NaN in the unreferenced
triangle and around B.  The residual |op(A) X - alpha B| stays below 4 m eps
|op(A)||X| per element (a backward-stable solve; well-conditioned triangles, so
the block inverses add at most a small factor).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("m,n", [(m, n) for m in (1, 63, 64, 65, 130, 192, 255, 256, 257, 300, 600) for n in (1, 15, 17, 100)]
                         + [(65, 8200), (256, 8200), (300, 8200)])
def test_trsm_left(oba, dt, m, n):
    L = oba.lib()
    rng = np.random.default_rng(n * 31 + m)
    eps = np.finfo(dt).eps
    f = L.cblas_dtrsm if dt == np.float64 else L.cblas_strsm
    B = rng.standard_normal((n, m + 3)).astype(dt)      # row j = column j
    B[:, m:] = np.nan
    dB = oba.DeviceBuffer(B.nbytes)
    for lower in (0, 1):
        for trans in (0, 1):
            for unit in (0, 1):
                T = rng.standard_normal((m, m))
                T = np.tril(T, -1) if lower else np.triu(T, 1)
                T /= 2 * np.sqrt(m)
                d = rng.uniform(1, 2, m)
                A = (T + np.diag(np.full(m, np.nan) if unit else d)).astype(dt)
                A[~np.tril(np.ones((m, m), bool)) if lower else ~np.triu(np.ones((m, m), bool))] = np.nan
                buf = np.full((m, m + 1), np.nan, dt)   # odd leading dimension
                buf[:, :m] = A.T
                dA = oba.DeviceBuffer.from_array(buf)
                L.openblas_amd_memcpy(dB.ptr, B.ctypes.data, B.nbytes, 0)
                f(102, 141, 122 if lower else 121, 112 if trans else 111, 132 if unit else 131, m, n, 0.5, dA.ptr,
                  m + 1, dB.ptr, m + 3)
                X = dB.to_array(np.empty_like(B))
                assert np.isnan(X[:, m:]).all()
                M = T.astype(dt).astype(np.float64) + np.diag(np.ones(m) if unit else d.astype(dt).astype(np.float64))
                M = M.T if trans else M
                x = X[:, :m].T.astype(np.float64)
                R = M @ x - 0.5 * B[:, :m].T.astype(np.float64)
                bound = 4 * m * eps * (np.abs(M) @ np.abs(x) + np.abs(B[:, :m].T))
                assert np.all(np.abs(R) <= bound), (lower, trans, unit, float((np.abs(R) / bound).max()))
