"""Scheme II's INT8 GEMM over its 128-deep slabs: K of one to five slabs and
around them, so both buffers are overwritten, in both tile sizes, and the large
tile with a K of more than one chunk of 16384, whose residues accumulate.
Integer operands, so the products are exact."""
import numpy as np
import pytest

from test_gpu_ozaki2_tiles import _exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(1, 1), (16, 130), (131, 255), (257, 260)])
@pytest.mark.parametrize("k", [127, 255, 256, 257, 384, 513])
def test_small_tiles(oba, m, n, k):
    _exact(oba, m, n, k, 0, 16, m + n + k)


@pytest.mark.parametrize("m,n,k", [(4090, 4097, 257), (4096, 4096, 400), (4081, 4090, 641)])
def test_large_tiles(oba, m, n, k):
    _exact(oba, m, n, k, 0, 12, k)


def test_large_tiles_two_chunks(oba):
    m = n = 4096
    k = 16384 + 130
    rng = np.random.default_rng(k)
    a = np.asfortranarray(rng.integers(-8, 9, (m, k)).astype(np.float64))
    b = np.asfortranarray(rng.integers(-8, 9, (k, n)).astype(np.float64))
    dA, dB, dC = oba.DeviceBuffer.from_array(a), oba.DeviceBuffer.from_array(b), oba.DeviceBuffer(8 * m * n)
    nm = oba.lib().openblas_amd_dgemm_ozaki2(102, 111, 111, m, n, k, 1.0, dA.ptr, m, dB.ptr, k, 0.0, dC.ptr, m, 0)
    assert nm > 0
    c = dC.to_array(np.empty((m, n), order="F"))
    rows = np.r_[0:20, 120:140, 250:262, 2040:2060, m - 20:m]
    assert np.array_equal(c[rows], a[rows] @ b)
