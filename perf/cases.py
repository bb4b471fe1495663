"""The calls whose speed is tracked, through the C ABI of libopenblas_amd with
operands resident in device memory (column-major, as a BLAS caller holds them).

A case names the routine and its arguments.  A matrix of m x n with leading
dimension ld is a torch tensor of shape (n, ld): row j of the tensor is column
j of the matrix.  Routines that overwrite their input get it restored from a
pristine copy inside every pass (openblas_amd_memcpy), so each pass does the
same work and returns the same values.
"""
import ctypes
import math

import numpy as np
import torch

import openblas_amd as oa

_DT = {"d": torch.float64, "s": torch.float32}
_C = {"d": ctypes.c_double, "s": ctypes.c_float}


def listed():
    return [
        # one small product: the call's fixed cost (checks, launch, completion)
        {"name": "dgemm_64", "op": "gemm", "dt": "d", "ta": False, "tb": False, "m": 64, "n": 64, "k": 64,
         "pad": 0, "alpha": 1.0, "beta": 0.0},
        # a small product with odd sizes and odd leading dimensions, as slices of a user's arrays have
        {"name": "sgemm_odd_small", "op": "gemm", "dt": "s", "ta": False, "tb": True, "m": 333, "n": 257, "k": 411,
         "pad": 4, "alpha": 1.0, "beta": 0.0},
        # the classic square benchmark size, about one output tile per CU
        {"name": "dgemm_1024", "op": "gemm", "dt": "d", "ta": False, "tb": False, "m": 1024, "n": 1024, "k": 1024,
         "pad": 0, "alpha": 1.0, "beta": 0.0},
        # an accumulating update C -= A^T B with odd sizes
        {"name": "dgemm_odd", "op": "gemm", "dt": "d", "ta": True, "tb": False, "m": 2047, "n": 3001, "k": 1501,
         "pad": 0, "alpha": -1.0, "beta": 1.0},
        # the large square product
        {"name": "sgemm_8192", "op": "gemm", "dt": "s", "ta": False, "tb": False, "m": 8192, "n": 8192, "k": 8192,
         "pad": 0, "alpha": 1.0, "beta": 0.0},
        # solving many right-hand sides with a triangular factor
        {"name": "dtrsm_8192x1024", "op": "trsm", "dt": "d", "side": "L", "uplo": "L", "trans": False, "unit": False,
         "m": 8192, "n": 1024},
        # a dense FP64 system of ordinary, odd size
        {"name": "dgesv_5001", "op": "gesv", "n": 5001, "nrhs": 3},
        # the mixed-precision solve of a large system (FP32 factors, FP64 refinement)
        {"name": "dsgesv_16384", "op": "dsgesv", "n": 16384, "nrhs": 1, "kappa": 100.0},
        # factoring a large covariance-like matrix
        {"name": "dpotrf_8192", "op": "potrf", "dt": "d", "uplo": "L", "n": 8192},
        # many small products of uneven size in one call
        {"name": "dgemm_batch_10000", "op": "gemm_batch", "dt": "d", "count": 10000, "lo": 8, "hi": 256,
         "square": True},
        # many small factorizations of uneven size in one call
        {"name": "dgetrf_batch_10000", "op": "getrf_batch", "dt": "d", "count": 10000, "lo": 8, "hi": 256},
        # the large FP64 product computed on the INT8 matrix cores, on data with some exponent spread
        {"name": "ozaki2_8192", "op": "ozaki2", "m": 8192, "n": 8192, "k": 8192, "phi": 0.5},
    ]


def _size(rng, lo, hi):
    """log-uniform; a quarter of the draws on a multiple of 64"""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.25:
        v = max(lo, (v + 32) // 64 * 64) if v >= 64 else v
    return min(max(v, lo), hi)


def draw(rng):
    op = rng.choice(["gemm", "gemm", "gemm", "gemm", "trsm", "trsm", "gesv", "dsgesv", "potrf", "gemm_batch",
                     "getrf_batch", "ozaki2"])
    if op == "gemm":
        return {"op": op, "dt": rng.choice("ds"), "ta": rng.random() < 0.5, "tb": rng.random() < 0.5,
                "m": _size(rng, 24, 8192), "n": _size(rng, 24, 8192), "k": _size(rng, 24, 8192),
                "pad": rng.choice([0, 0, 1, 4, 7]), "alpha": rng.choice([1.0, -1.0, 0.7]),
                "beta": rng.choice([0.0, 0.0, 1.0])}
    if op == "trsm":
        side = rng.choice("LR")
        a, b = _size(rng, 200, 8192), _size(rng, 64, 4096)
        return {"op": op, "dt": rng.choice("ds"), "side": side, "uplo": rng.choice("LU"), "trans": rng.random() < 0.5,
                "unit": rng.random() < 0.3, "m": a if side == "L" else b, "n": b if side == "L" else a}
    if op == "gesv":
        return {"op": op, "n": _size(rng, 300, 6000), "nrhs": rng.randint(1, 40)}
    if op == "dsgesv":
        return {"op": op, "n": _size(rng, 1000, 12000), "nrhs": rng.randint(1, 16), "kappa": 100.0}
    if op == "potrf":
        return {"op": op, "dt": rng.choice("ds"), "uplo": rng.choice("LLU"), "n": _size(rng, 500, 9000)}
    if op == "gemm_batch":
        return {"op": op, "dt": rng.choice("ds"), "count": _size(rng, 300, 10000), "lo": rng.randint(4, 16),
                "hi": rng.randint(60, 256), "square": rng.random() < 0.5}
    if op == "getrf_batch":
        return {"op": op, "dt": "d", "count": _size(rng, 300, 10000), "lo": rng.randint(4, 16),
                "hi": rng.randint(60, 256)}
    return {"op": op, "m": _size(rng, 1500, 8192), "n": _size(rng, 1500, 8192), "k": _size(rng, 1000, 8192),
            "phi": rng.choice([0.5, 1.0])}


# ---- inputs -----------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, dt=torch.float64):
    return torch.randn(*shape, generator=g, device="cuda", dtype=dt)


def _rand(g, *shape, dt=torch.float64):
    return torch.rand(*shape, generator=g, device="cuda", dtype=dt)


def _system(g, n, kappa):
    """A = Q1 diag(s) Q2, the Qs products of 8 Householder reflectors, s
    geometric from 1 to 1/kappa; as a tensor of A's columns"""
    s = kappa ** (-torch.arange(n, device="cuda", dtype=torch.float64) / (n - 1))
    a = torch.diag(s)
    for _ in range(8):
        v = _randn(g, n)
        v /= v.norm()
        a.addr_(v, torch.mv(a.t(), v), alpha=-2.0)
        w = _randn(g, n)
        w /= w.norm()
        a.addr_(torch.mv(a, w), w, alpha=-2.0)
    return a


def _triangle(g, n, uplo, unit, dt):
    """the Cholesky factor of a Wishart matrix with 2n degrees of freedom
    (Bartlett: normal off the diagonal, about chi on it); unit: its L D L^T
    form.  The other triangle holds other numbers, which a solve ignores."""
    t = _randn(g, n, n, dt=dt)
    d = torch.sqrt(2.0 * n - torch.arange(n, device="cuda", dtype=dt))
    if unit:   # columns of L (rows of U) divided by the diagonal
        t /= d[:, None] if uplo == "L" else d[None, :]
    t.diagonal().copy_(d)
    return t


def _sizes(case, fields):
    """the batch's uneven sizes, uniform in lo..hi: part of the case, not of its data"""
    r = np.random.default_rng((case["count"], case["lo"], case["hi"]))
    n = r.integers(case["lo"], case["hi"] + 1, (fields, case["count"]))
    return n.astype(np.int32)


def _offsets(counts):
    o = np.zeros(len(counts), np.int64)
    o[1:] = np.cumsum(counts.astype(np.int64))[:-1]
    return o


def _ptrs(base, off, es):
    return np.ascontiguousarray(base + off * es, dtype=np.uint64)


def _cp(a, ty):
    return a.ctypes.data_as(ctypes.POINTER(ty))


def _gemm_batch_sizes(case):
    if case["square"]:
        n = _sizes(case, 1)[0]
        return n, n, n
    return tuple(np.ascontiguousarray(v) for v in _sizes(case, 3))


def prepare(case, seed):
    op = case["op"]
    g = _gen(seed)
    st = {"case": case, "L": oa.lib()}
    if op == "gemm":
        dt = _DT[case["dt"]]
        m, n, k, pad = case["m"], case["n"], case["k"], case["pad"]
        st["lda"], st["ldb"], st["ldc"] = (k if case["ta"] else m) + pad, (n if case["tb"] else k) + pad, m + pad
        st["a"] = _rand(g, m if case["ta"] else k, st["lda"], dt=dt) * 2 - 1
        st["b"] = _rand(g, k if case["tb"] else n, st["ldb"], dt=dt) * 2 - 1
        if case["beta"] != 0.0:
            st["c0"] = _rand(g, n, st["ldc"], dt=dt) * 2 - 1
            st["c"] = st["c0"].clone()
        else:
            st["c"] = torch.zeros(n, st["ldc"], device="cuda", dtype=dt)
    elif op == "trsm":
        dt = _DT[case["dt"]]
        na = case["m"] if case["side"] == "L" else case["n"]
        st["a"] = _triangle(g, na, case["uplo"], case["unit"], dt)
        st["b0"] = _randn(g, case["n"], case["m"], dt=dt)
        st["b"] = st["b0"].clone()
    elif op in ("gesv", "dsgesv"):
        n, nrhs = case["n"], case["nrhs"]
        st["a0"] = _randn(g, n, n) if op == "gesv" else _system(g, n, case["kappa"])
        st["b0"] = _randn(g, nrhs, n)
        st["a"] = st["a0"].clone()
        st["b"] = st["b0"].clone()
        st["ipiv"] = torch.zeros(n, device="cuda", dtype=torch.int32)
        st["n"], st["nrhs"] = ctypes.c_int(n), ctypes.c_int(nrhs)
        st["info"], st["iter"] = ctypes.c_int(-1), ctypes.c_int(-99)
        if op == "dsgesv":
            st["x"] = torch.zeros(nrhs, n, device="cuda", dtype=torch.float64)
    elif op == "potrf":
        n, dt = case["n"], _DT[case["dt"]]
        z = _randn(g, n, n, dt=dt)
        st["a0"] = torch.mm(z, z.t()).div_(n)   # sample covariance, regularised
        st["a0"].diagonal().add_(0.1)
        st["a"] = st["a0"].clone()
        st["n"], st["info"] = ctypes.c_int(n), ctypes.c_int(-1)
    elif op == "gemm_batch":
        dt, ty, es = _DT[case["dt"]], _C[case["dt"]], 8 if case["dt"] == "d" else 4
        m, n, k = _gemm_batch_sizes(case)
        count = case["count"]
        ca, cb, cc = (x.astype(np.int64) * y for x, y in ((m, k), (k, n), (m, n)))
        st["a"] = _randn(g, int(ca.sum()), dt=dt)
        st["b"] = _randn(g, int(cb.sum()), dt=dt)
        st["c"] = torch.zeros(int(cc.sum()), device="cuda", dtype=dt)
        keep = {
            "t": np.full(count, oa.NoTrans, np.int32), "m": m, "n": n, "k": k,
            "alpha": np.ones(count, np.float64 if es == 8 else np.float32),
            "beta": np.zeros(count, np.float64 if es == 8 else np.float32),
            "pa": _ptrs(st["a"].data_ptr(), _offsets(ca), es), "pb": _ptrs(st["b"].data_ptr(), _offsets(cb), es),
            "pc": _ptrs(st["c"].data_ptr(), _offsets(cc), es), "size": np.ones(count, np.int32)}
        st["keep"] = keep
        ci, vp = ctypes.c_int, ctypes.c_void_p
        st["args"] = (oa.ColMajor, _cp(keep["t"], ci), _cp(keep["t"], ci), _cp(m, ci), _cp(n, ci), _cp(k, ci),
                      _cp(keep["alpha"], ty), _cp(keep["pa"], vp), _cp(m, ci), _cp(keep["pb"], vp), _cp(k, ci),
                      _cp(keep["beta"], ty), _cp(keep["pc"], vp), _cp(m, ci), count, _cp(keep["size"], ci))
    elif op == "getrf_batch":
        n = np.ascontiguousarray(_sizes(case, 1)[0])
        count, c2 = case["count"], n.astype(np.int64) ** 2
        st["a0"] = _randn(g, int(c2.sum()))
        st["a"] = st["a0"].clone()
        st["ipiv"] = torch.zeros(int(n.sum()), device="cuda", dtype=torch.int32)
        keep = {"n": n, "pa": _ptrs(st["a"].data_ptr(), _offsets(c2), 8),
                "pp": _ptrs(st["ipiv"].data_ptr(), _offsets(n), 4), "info": np.full(count, -1, np.int32)}
        st["keep"] = keep
        ci, vp = ctypes.c_int, ctypes.c_void_p
        st["args"] = (_cp(n, ci), _cp(n, ci), _cp(keep["pa"], vp), _cp(n, ci), _cp(keep["pp"], vp),
                      _cp(keep["info"], ci), count)
    else:
        m, n, k = case["m"], case["n"], case["k"]
        st["a"] = (_rand(g, k, m) - 0.5) * torch.exp(case["phi"] * _randn(g, k, m))
        st["b"] = (_rand(g, n, k) - 0.5) * torch.exp(case["phi"] * _randn(g, n, k))
        st["c"] = torch.zeros(n, m, device="cuda", dtype=torch.float64)
    torch.cuda.synchronize()   # the library runs on a stream of its own
    return st


# ---- one pass ---------------------------------------------------------------------
def _restore(st, dst, src):
    st["L"].openblas_amd_memcpy(st[dst].data_ptr(), st[src].data_ptr(), st[src].numel() * st[src].element_size(), 2)


def run(st):
    case, L = st["case"], st["L"]
    op = case["op"]
    if op == "gemm":
        if "c0" in st:
            _restore(st, "c", "c0")
        f = L.cblas_dgemm if case["dt"] == "d" else L.cblas_sgemm
        f(oa.ColMajor, oa.Trans if case["ta"] else oa.NoTrans, oa.Trans if case["tb"] else oa.NoTrans, case["m"],
          case["n"], case["k"], case["alpha"], st["a"].data_ptr(), st["lda"], st["b"].data_ptr(), st["ldb"],
          case["beta"], st["c"].data_ptr(), st["ldc"])
        return st["c"]
    if op == "trsm":
        _restore(st, "b", "b0")
        f = L.cblas_dtrsm if case["dt"] == "d" else L.cblas_strsm
        na = case["m"] if case["side"] == "L" else case["n"]
        f(oa.ColMajor, oa.Left if case["side"] == "L" else oa.Right, oa.Lower if case["uplo"] == "L" else oa.Upper,
          oa.Trans if case["trans"] else oa.NoTrans, oa.Unit if case["unit"] else oa.NonUnit, case["m"], case["n"],
          1.0, st["a"].data_ptr(), na, st["b"].data_ptr(), case["m"])
        return st["b"]
    if op == "gesv":
        _restore(st, "a", "a0")
        _restore(st, "b", "b0")
        L.dgesv_(st["n"], st["nrhs"], st["a"].data_ptr(), st["n"], st["ipiv"].data_ptr(), st["b"].data_ptr(), st["n"],
                 st["info"])
        return {"x": st["b"], "lu": st["a"], "ipiv": st["ipiv"], "info": st["info"].value}
    if op == "dsgesv":
        # A stays as it is when the refinement converges; IPIV is of the FP32
        # factorization, whose near-ties depend on its summation order
        L.dsgesv_(st["n"], st["nrhs"], st["a"].data_ptr(), st["n"], st["ipiv"].data_ptr(), st["b"].data_ptr(), st["n"],
                  st["x"].data_ptr(), st["n"], None, None, st["iter"], st["info"])
        return {"x": st["x"], "iter": st["iter"].value, "info": st["info"].value}
    if op == "potrf":
        _restore(st, "a", "a0")
        f = L.dpotrf_ if case["dt"] == "d" else L.spotrf_
        f(case["uplo"].encode(), st["n"], st["a"].data_ptr(), st["n"], st["info"])
        return {"factor": st["a"], "info": st["info"].value}
    if op == "gemm_batch":
        (L.cblas_dgemm_batch if case["dt"] == "d" else L.cblas_sgemm_batch)(*st["args"])
        return st["c"]
    if op == "getrf_batch":
        _restore(st, "a", "a0")
        L.openblas_amd_dgetrf_batch(*st["args"])
        return {"lu": st["a"], "ipiv": st["ipiv"], "info": st["keep"]["info"]}
    moduli = L.openblas_amd_dgemm_ozaki2(oa.ColMajor, oa.NoTrans, oa.NoTrans, case["m"], case["n"], case["k"], 1.0,
                                         st["a"].data_ptr(), case["m"], st["b"].data_ptr(), case["k"], 0.0,
                                         st["c"].data_ptr(), case["m"], 0)
    return {"c": st["c"], "moduli": moduli}


# ---- the work of one pass -------------------------------------------------------------
def work(case):
    op = case["op"]
    es = 4 if case.get("dt") == "s" else 8
    if op == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": es * (m * k + k * n + m * n * (2 if case["beta"] else 1)), "flops": 2.0 * m * n * k}
    if op == "trsm":
        m, n = case["m"], case["n"]
        na = m if case["side"] == "L" else n
        return {"bytes": es * (na * na / 2 + 2 * m * n), "flops": 1.0 * na * m * n}
    if op == "gesv":
        n, r = case["n"], case["nrhs"]
        return {"bytes": es * (2.0 * n * n + 2.0 * n * r), "flops": 2.0 / 3.0 * n ** 3 + 2.0 * n * n * r}
    if op == "dsgesv":
        n, r = case["n"], case["nrhs"]
        return {"bytes": es * (1.0 * n * n + 2.0 * n * r), "flops": 2.0 / 3.0 * n ** 3 + 2.0 * n * n * r}
    if op == "potrf":
        n = case["n"]
        return {"bytes": es * 1.0 * n * n, "flops": n ** 3 / 3.0}
    lo, hi, c = case.get("lo", 0), case.get("hi", 0), case.get("count", 0)
    s = np.arange(lo, hi + 1, dtype=np.float64)
    m1, m2, m3 = (float((s ** p).mean()) for p in (1, 2, 3))
    if op == "gemm_batch":
        if case["square"]:
            return {"bytes": es * 3 * m2 * c, "flops": 2 * m3 * c}
        return {"bytes": es * 3 * m1 * m1 * c, "flops": 2 * m1 ** 3 * c}
    if op == "getrf_batch":
        return {"bytes": 2 * es * m2 * c, "flops": 2.0 / 3.0 * m3 * c}
    m, n, k = case["m"], case["n"], case["k"]
    return {"bytes": es * (m * k + k * n + m * n), "flops": 2.0 * m * n * k}


# ---- the same values from plain torch in 64 bits -----------------------------------------
def exact(case, seed):
    op = case["op"]
    st = prepare(case, seed)
    if op == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        a = st["a"][:, :k].double() if case["ta"] else st["a"][:, :m].double().t()    # m x k
        b = st["b"][:, :n].double().t() if case["tb"] else st["b"][:, :k].double()    # n x k
        c = st["c0"].double() if "c0" in st else st["c"].double()
        c[:, :m] = case["alpha"] * torch.mm(b, a.t()) + case["beta"] * c[:, :m]
        return c
    if op == "trsm":
        t = st["a"].double().t()   # the matrix itself
        upper = case["uplo"] == "U"
        t = t.triu() if upper else t.tril()
        b = st["b0"].double().t()
        if case["trans"]:
            t, upper = t.t(), not upper
        x = torch.linalg.solve_triangular(t.cpu(), b.cpu(), upper=upper, left=case["side"] == "L",
                                          unitriangular=case["unit"])
        return x.t().contiguous()
    if op == "gesv":
        a, b = st["a0"].cpu().t(), st["b0"].cpu().t()
        lu, piv = torch.linalg.lu_factor(a)
        return {"x": torch.linalg.lu_solve(lu, piv, b).t().contiguous(), "lu": lu.t().contiguous(), "ipiv": None,
                "info": None}
    if op == "dsgesv":
        x = torch.linalg.solve(st["a0"].cpu().t(), st["b0"].cpu().t())
        return {"x": x.t().contiguous(), "iter": None, "info": None}
    if op == "potrf":
        a = st["a0"].double().t().cpu()
        f = torch.linalg.cholesky(a, upper=case["uplo"] == "U")
        f = f.tril() + a.triu(1) if case["uplo"] == "L" else f.triu() + a.tril(-1)
        return {"factor": f.t().contiguous(), "info": None}
    if op == "gemm_batch":
        m, n, k = _gemm_batch_sizes(case)
        a, b = st["a"].double().cpu().numpy(), st["b"].double().cpu().numpy()
        out, oa_, ob = [], 0, 0
        for mi, ni, ki in zip(m.tolist(), n.tolist(), k.tolist()):
            x, y = a[oa_:oa_ + mi * ki].reshape(ki, mi), b[ob:ob + ki * ni].reshape(ni, ki)
            out.append((y @ x).reshape(-1))
            oa_, ob = oa_ + mi * ki, ob + ki * ni
        return np.concatenate(out)
    if op == "getrf_batch":
        a, out, o = st["a0"].cpu(), [], 0
        for n in st["keep"]["n"].tolist():
            lu, _ = torch.linalg.lu_factor(a[o:o + n * n].reshape(n, n).t())
            out.append(lu.t().reshape(-1))
            o += n * n
        return {"lu": torch.cat(out), "ipiv": None, "info": None}
    return {"c": torch.mm(st["b"], st["a"]), "moduli": None}
