"""Scheme II at the edges of its INT8 GEMM tiles (128 and, for large products,
256 wide), of its 64-deep slabs (1, 2, 3 and more), of its k chunks of 16384 and
of its operand pieces (many moduli): integer operands, whose products FP64 holds
exactly, come out exactly, and rows past C keep their bits.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _exact(oba, m, n, k, moduli, bits, seed):
    rng = np.random.default_rng(seed)
    a = np.asfortranarray(rng.integers(-(1 << bits), (1 << bits) + 1, (m, k)).astype(np.float64))
    b = np.asfortranarray(rng.integers(-(1 << bits), (1 << bits) + 1, (k, n)).astype(np.float64))
    c = np.full((m + 3, n), 7.5, order="F")
    nm = oba.lib().openblas_amd_dgemm_ozaki2(102, 111, 111, m, n, k, 1.0, a.ctypes.data, m, b.ctypes.data, k, 0.0,
                                             c.ctypes.data, m + 3, moduli)
    assert nm > 0
    assert np.array_equal(c[:m], a @ b), (m, n, k, moduli)
    assert np.all(c[m:] == 7.5)


@pytest.mark.parametrize("m,n", [(1, 1), (15, 17), (16, 130), (127, 129), (128, 128), (131, 255), (257, 260)])
@pytest.mark.parametrize("k", [1, 63, 64, 65, 128, 129, 200])
def test_ozaki2_small_tiles(oba, m, n, k):
    _exact(oba, m, n, k, 0, 16, m + n + k)


@pytest.mark.parametrize("m,n,k", [(4090, 4097, 64), (4096, 4096, 100), (4081, 4090, 190)])
def test_ozaki2_large_tiles(oba, m, n, k):
    _exact(oba, m, n, k, 0, 12, k)


@pytest.mark.parametrize("k", [16383, 16384, 16385, 32768, 40000])
def test_ozaki2_k_chunks(oba, k):
    _exact(oba, 20, 33, k, 0, 14, k)


@pytest.mark.parametrize("moduli", [9, 13, 20, 25, 30])
def test_ozaki2_pieces(oba, moduli):
    _exact(oba, 70, 40, 90, moduli, 20, moduli)
