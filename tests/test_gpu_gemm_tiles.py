"""GEMM at the edges of its tiles: sizes one off the 32/64/128 tile and the
slab depths, operands narrower than a tile, odd leading dimensions and operands
that start at an element-aligned but not 16-byte-aligned device address, the
split and sliced K ranges, and C's surroundings untouched.  Compared with the
FP64 product; the tolerance is the ctest dmmch bound of 16 times
eps * (|alpha| |A||B| + |beta||C|) per element.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TR = {0: 111, 1: 112}

SHAPES = [(1, 1, 1), (31, 33, 7), (32, 32, 16), (33, 31, 17), (63, 65, 9), (64, 64, 8), (65, 129, 33), (5, 300, 65),
          (300, 5, 65), (257, 31, 129), (70, 90, 1025), (130, 66, 4100),        # 32x32 tiles, split K
          (1023, 961, 511), (1024, 1024, 513), (961, 1024, 530),                # about one 64x64 tile per CU
          (1030, 1090, 70), (1999, 2001, 37)]                                   # more tiles than CUs


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_tile_edges(oba, dt, m, n, k, ta, tb):
    L = oba.lib()
    rng = np.random.default_rng(m * 7 + n * 3 + k + 2 * ta + tb)
    es = np.dtype(dt).itemsize
    eps = np.finfo(dt).eps
    alpha, beta = (1.0, 0.0) if (m + n + k) % 2 else (-0.7, 1.3)
    ar, ac, br, bc = (k if ta else m), (m if ta else k), (n if tb else k), (k if tb else n)
    lda, ldb, ldc, off = ar + 1, br + 3, m + 5, 1     # one element past the allocation's start
    A = rng.uniform(-1, 1, (ac, lda)).astype(dt)      # row j = column j of the matrix
    B = rng.uniform(-1, 1, (bc, ldb)).astype(dt)
    C = rng.uniform(-1, 1, (n, ldc)).astype(dt)
    A[:, ar:], B[:, br:] = np.nan, np.nan             # outside the matrices
    bufs = [oba.DeviceBuffer.from_array(np.concatenate([np.full(off, np.nan, dt), X.ravel()])) for X in (A, B, C)]
    f = L.cblas_dgemm if dt == np.float64 else L.cblas_sgemm
    f(102, TR[ta], TR[tb], m, n, k, alpha, bufs[0].ptr + off * es, lda, bufs[1].ptr + off * es, ldb, beta,
      bufs[2].ptr + off * es, ldc)
    got = bufs[2].to_array(np.empty(off + C.size, dt))[off:].reshape(n, ldc)
    a = (A[:, :ar] if ta else A[:, :ar].T).astype(np.float64)        # m x k
    b = (B[:, :br] if tb else B[:, :br].T).astype(np.float64)        # k x n
    c0 = C[:, :m].T.astype(np.float64)
    al, be = float(dt(alpha)), float(dt(beta))
    ref = al * (a @ b) + be * c0
    g = abs(al) * (np.abs(a) @ np.abs(b)) + abs(be) * np.abs(c0)
    err = np.abs(got[:, :m].T.astype(np.float64) - ref)
    assert np.all(err <= 16 * eps * g), float((err / (eps * np.maximum(g, 1e-300))).max())
    assert np.array_equal(got[:, m:], C[:, m:])       # the rows past m
