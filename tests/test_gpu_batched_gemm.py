"""Batched GEMM at the edges of its 64- and 32-wide tiles and of its k slabs (8,
16 and 32 deep), all four transpose forms, padded leading dimensions: the exact
product within (k+2)*eps*(|alpha| |A||B| + |beta C|), which bounds any order of
summation and the two products with the scalars; padding untouched; a K tail
that overlaps the slab before must not let an infinity of one operand meet a
cleared element of the other.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(oba, dt, ta, tb, probs, alpha, beta):
    L = oba.lib()
    f = L.cblas_dgemm_batch if dt == np.float64 else L.cblas_sgemm_batch
    cnt = len(probs)
    ia = lambda v: (ctypes.c_int * len(v))(*v)
    pa = lambda v: (ctypes.c_void_p * len(v))(*v)
    sc = lambda v: np.full(cnt, v, dt)
    ct = ctypes.c_double if dt == np.float64 else ctypes.c_float
    al, be = (sc(v).ctypes.data_as(ctypes.POINTER(ct)) for v in (alpha, beta))
    f(102, ia([112 if ta else 111] * cnt), ia([112 if tb else 111] * cnt), ia([p["m"] for p in probs]),
      ia([p["n"] for p in probs]), ia([p["k"] for p in probs]), al, pa([p["a"].ctypes.data for p in probs]),
      ia([p["a"].shape[0] for p in probs]), pa([p["b"].ctypes.data for p in probs]), ia([p["b"].shape[0] for p in probs]),
      be, pa([p["c"].ctypes.data for p in probs]), ia([p["c"].shape[0] for p in probs]), cnt,
      ia([1] * cnt))


def _operand(rng, dt, r, c):
    a = np.asfortranarray(rng.standard_normal((max(r, 1) + int(rng.integers(0, 3)), max(c, 1))).astype(dt))
    return a


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_batch_edges(oba, dt, ta, tb):
    rng = np.random.default_rng(11 + 2 * ta + tb)
    dims = [1, 15, 31, 32, 33, 47, 63, 64, 65, 95, 96, 97, 127, 128, 129, 161]
    ks = [0, 1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 65, 100]
    probs = []
    for i, m in enumerate(dims):
        for j, n in enumerate(dims):
            k = ks[(5 * i + 3 * j) % len(ks)]
            probs.append({"m": m, "n": n, "k": k, "a": _operand(rng, dt, k if ta else m, m if ta else k),
                          "b": _operand(rng, dt, n if tb else k, k if tb else n), "c": _operand(rng, dt, m, n)})
    old = [p["c"].copy(order="F") for p in probs]
    _run(oba, dt, ta, tb, probs, 0.75, -0.5)
    eps = np.finfo(dt).eps
    for p, c0 in zip(probs, old):
        m, n, k = p["m"], p["n"], p["k"]
        a = (p["a"][:k, :m].T if ta else p["a"][:m, :k]).astype(np.float64)
        b = (p["b"][:n, :k].T if tb else p["b"][:k, :n]).astype(np.float64)
        want = 0.75 * a @ b - 0.5 * c0[:m]
        bound = (k + 2) * eps * (0.75 * np.abs(a) @ np.abs(b) + 0.5 * np.abs(c0[:m]))
        assert np.all(np.abs(p["c"][:m] - want) <= bound), (m, n, k)
        assert np.array_equal(p["c"][m:], c0[m:])


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_gemm_batch_tail_infinity(oba, dt):
    rng = np.random.default_rng(3)
    probs = []
    for m, n, k in ((64, 64, 37), (65, 130, 61), (33, 40, 37), (20, 70, 45), (64, 20, 45)):
        a, b = _operand(rng, dt, m, k), _operand(rng, dt, k, n)
        a[m // 2, k - 6] = np.inf      # in the last two slabs' common part
        b[k - 7, n // 2] = -np.inf
        probs.append({"m": m, "n": n, "k": k, "a": a, "b": b, "c": np.full((m, n), np.nan, dt, order="F")})
    _run(oba, dt, 0, 0, probs, 1.0, 0.0)
    for p in probs:
        m, n, k = p["m"], p["n"], p["k"]
        a, b = p["a"][:m, :k].astype(np.float64), p["b"][:k, :n].astype(np.float64)
        with np.errstate(invalid="ignore"):
            want = np.zeros((m, n))
            for q in range(k):
                want += np.outer(a[:, q], b[q])
        assert np.array_equal(np.isnan(p["c"]), np.isnan(want)) and np.array_equal(np.isinf(p["c"]), np.isinf(want))
        fin = np.isfinite(want)
        absf = np.where(np.isfinite(a), np.abs(a), 0) @ np.where(np.isfinite(b), np.abs(b), 0)
        assert np.all(np.abs(p["c"] - want)[fin] <= ((k + 2) * np.finfo(dt).eps * absf)[fin])
