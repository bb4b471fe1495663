"""Products of few tiles and a deep K, which is split over workgroups: the sizes
take every tile of the split (32x32 with four and two groups, 64x32, 64x64) and
the unsplit forms beside them, with K that leaves a short last part, odd leading
dimensions, all transpose forms.  |C - want| <= (k + 4) eps (|alpha| |A||B| +
|beta C|), which bounds any order of summation, the sum of the parts and the
products with the scalars; padding untouched, and beta = 0 reads no C."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(200, 130, 1030), (256, 256, 5003), (640, 256, 1500), (512, 640, 2051), (640, 640, 3001), (1280, 400, 1281),
         (1281, 637, 1301), (800, 1024, 1999), (100, 2700, 2048), (48, 2700, 4099), (2700, 33, 4099), (5440, 17, 2100),
         (5440, 32, 2047), (16, 5441, 2113), (31, 2700, 3000), (640, 1280, 1024), (1025, 770, 1279)]


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("m,n,k", SIZES)
def test_gemm_split(oba, dt, m, n, k):
    L = oba.lib()
    f = L.cblas_dgemm if dt == np.float64 else L.cblas_sgemm
    rng = np.random.default_rng(m + n + k)
    eps = np.finfo(dt).eps
    a0, b0 = rng.uniform(-1, 1, (m, k)).astype(dt), rng.uniform(-1, 1, (k, n)).astype(dt)
    prod = a0.astype(np.float64) @ b0.astype(np.float64)
    mag = np.abs(a0).astype(np.float64) @ np.abs(b0).astype(np.float64)
    for form, (ta, tb) in enumerate([(0, 0), (0, 1), (1, 0), (1, 1)]):
        beta = (0.0, -0.5)[form % 2]
        rows = lambda x, t: np.ascontiguousarray(x if t else x.T)   # row j: column j of the stored matrix
        a, b = rows(a0, ta), rows(b0, tb)
        pad = lambda x: np.concatenate([x, np.full((x.shape[0], 1), np.nan, dt)], axis=1)
        A, B = pad(a), pad(b)
        C = np.full((n, m + 1), np.nan, dt)
        c0 = rng.uniform(-1, 1, (n, m)).astype(dt)
        if beta != 0.0:
            C[:, :m] = c0
        dA, dB, dC = (oba.DeviceBuffer.from_array(x) for x in (A, B, C))
        f(102, 112 if ta else 111, 112 if tb else 111, m, n, k, 0.75, dA.ptr, A.shape[1], dB.ptr, B.shape[1], beta,
          dC.ptr, m + 1)
        got = dC.to_array(np.empty_like(C))
        assert np.isnan(got[:, m]).all()
        want = 0.75 * prod + beta * c0.T.astype(np.float64)
        bound = (k + 4) * eps * (0.75 * mag + abs(beta) * np.abs(c0.T))
        assert np.all(np.abs(got[:, :m].T - want) <= bound), (ta, tb)
