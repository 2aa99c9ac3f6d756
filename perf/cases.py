"""Performance cases of the dense LU solve path.

Each case is one pass through the public entry points of `lapack_amd` as a
program uses them: factor and solve on arrays in GPU memory (the synchronous
drop-in and the stream-ordered form), the drop-in on host arrays, FP64, FP32
and mixed precision, repeated solves on saved factors, batches of systems of
uneven order, and the adjoint of a batch.

Matrices are column-major: the tensor t of shape (n, m) holds the m x n matrix
A(i, j) = t[j, i].  FP64 matrices are N(0,1), as the benchmark's.  Matrices
that are factored in FP32 are well conditioned with their equations in no
particular order (a permuted diagonal of 2 over N(0,1)/sqrt(n) entries), the
systems for which single precision is used: every pivot search finds a row to
interchange, and the pivots do not hinge on the last bits.
"""
import numpy as np
import torch

import lapack_amd as la

DEV = "cuda"


def listed():
    return [
        # one small solve behind a synchronous call: latency and launches
        {"name": "gesv_n100", "op": "gesv", "n": 100, "nrhs": 1},
        # a Fortran or numpy program's call: operands in host memory
        {"name": "gesv_host_n500", "op": "gesv_host", "n": 500, "nrhs": 4},
        # the reference-sized solve of the benchmark (n = 1024, one right-hand side)
        {"name": "lu_n1024", "op": "lu", "n": 1024, "nrhs": 1},
        # an ordinary order, a power of two and a ragged one
        {"name": "lu_n4096", "op": "lu", "n": 4096, "nrhs": 16},
        # the benchmark's headline order
        {"name": "lu_n16384", "op": "lu", "n": 16384, "nrhs": 16},
        # a tall block, as a panel of a larger factorization: odd sizes, lda > m
        {"name": "getrf_9001x1201", "op": "getrf", "m": 9001, "n": 1201, "lda": 9008},
        # single precision
        {"name": "lu_f32_n1500", "op": "lu_f32", "n": 1500, "nrhs": 3},
        # FP32 factorization, FP64 accuracy
        {"name": "dsgesv_n8192", "op": "dsgesv", "n": 8192, "nrhs": 1},
        # saved factors, many solves: one right-hand side against A^T
        {"name": "getrs_t_n6001", "op": "getrs", "trans": "T", "n": 6001, "nrhs": 1},
        # the benchmark's batch: 10000 systems of uneven order, FP64
        {"name": "batch_f64", "op": "batch", "prec": "d", "batch": 10000, "lo": 16, "hi": 512},
        # a smaller batch of small systems, FP32
        {"name": "batch_f32", "op": "batch", "prec": "s", "batch": 3000, "lo": 8, "hi": 160},
        # the backward pass of the benchmark's 256 systems of order 1024
        {"name": "adjoint_256x1024", "op": "adjoint", "batch": 256, "n": 1024, "nrhs": 8},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    op = rng.choice(["gesv", "gesv_host", "lu", "lu", "lu", "getrf", "lu_f32", "dsgesv", "getrs", "batch", "batch",
                     "adjoint"])
    if op == "gesv":
        return {"op": op, "n": _log(rng, 16, 700), "nrhs": rng.randint(1, 8)}
    if op == "gesv_host":
        return {"op": op, "n": _log(rng, 50, 2000), "nrhs": rng.randint(1, 8)}
    if op == "lu":
        return {"op": op, "n": _log(rng, 150, 16000), "nrhs": rng.choice([1, 2, 3, 5, 8, 16, 24])}
    if op == "getrf":
        m, n = _log(rng, 200, 10000), _log(rng, 200, 10000)
        return {"op": op, "m": m, "n": n, "lda": m + rng.choice([0, 0, 1, 7, 64])}
    if op == "lu_f32":
        return {"op": op, "n": _log(rng, 100, 4096), "nrhs": rng.choice([1, 2, 3, 5, 16])}
    if op == "dsgesv":
        return {"op": op, "n": _log(rng, 300, 8192), "nrhs": rng.choice([1, 1, 2, 4])}
    if op == "getrs":
        return {"op": op, "trans": rng.choice(["N", "T"]), "n": _log(rng, 200, 12000),
                "nrhs": rng.choice([1, 2, 4, 7, 16, 32])}
    if op == "batch":
        lo = rng.choice([4, 8, 16, 33])
        return {"op": op, "prec": rng.choice(["d", "s"]), "batch": _log(rng, 64, 6000), "lo": lo,
                "hi": _log(rng, lo + 8, 512)}
    return {"op": "adjoint", "batch": _log(rng, 8, 200), "n": _log(rng, 64, 1024), "nrhs": rng.randint(1, 16)}


# ---- inputs -------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, *shape, dtype=torch.float64):
    return torch.randn(*shape, generator=g, device=DEV, dtype=dtype)


def _shuffled(g, n, dtype):
    """Well-conditioned matrix with its rows in random order, column-major."""
    t = _randn(g, n, n, dtype=dtype) / n ** 0.5
    t += 2.0 * torch.eye(n, device=DEV, dtype=dtype)
    return t[:, torch.randperm(n, generator=g, device=DEV)].contiguous()


def _batch_sizes(case):
    """Orders and right-hand-side counts: the same for every seed."""
    r = np.random.default_rng(case["batch"])
    ns = r.integers(case["lo"], case["hi"] + 1, case["batch"])
    nrhs = r.integers(1, 5, case["batch"])
    aoff = np.concatenate([[0], np.cumsum(ns * ns)])
    boff = np.concatenate([[0], np.cumsum(ns * nrhs)])
    return ns, nrhs, aoff, boff


def _batch_data(case, seed):
    """All matrices of the batch in one flat tensor, all right-hand sides in another."""
    ns, nrhs, aoff, boff = _batch_sizes(case)
    g = _gen(seed)
    dt = torch.float64 if case["prec"] == "d" else torch.float32
    if case["prec"] == "d":
        a = torch.rand(int(aoff[-1]), generator=g, device=DEV, dtype=dt) * 2 - 1
    else:
        # the well-conditioned form, matrix by matrix: element e of system k
        # is (i, j); column j carries its diagonal in row (j + shift) mod n
        nt = torch.from_numpy(ns).to(DEV)
        k = torch.repeat_interleave(torch.arange(len(ns), device=DEV), nt * nt)
        e = torch.arange(int(aoff[-1]), device=DEV) - torch.from_numpy(aoff[:-1]).to(DEV)[k]
        nk = nt[k]
        i, j = e % nk, e // nk
        shift = torch.randint(1, 1 << 20, (len(ns),), generator=g, device=DEV)
        a = torch.randn(int(aoff[-1]), generator=g, device=DEV, dtype=dt) / nk.to(dt).sqrt()
        a += 2.0 * (i == (j + shift[k]) % nk).to(dt)
    b = torch.rand(int(boff[-1]), generator=g, device=DEV, dtype=dt) * 2 - 1
    return ns, nrhs, aoff, boff, a, b


def _adjoint_data(case, seed):
    nb, n, r = case["batch"], case["n"], case["nrhs"]
    g = _gen(seed)
    a = _randn(g, nb, n, n)
    a += 4.0 * n ** 0.5 * torch.eye(n, device=DEV, dtype=torch.float64)
    return a, _randn(g, nb, r, n), _randn(g, nb, r, n)


def _data(case, seed):
    op = case["op"]
    g = _gen(seed)
    n = case["n"]
    if op == "getrf":
        return (_randn(g, n, case["lda"]),)
    if op == "lu_f32":
        a = _shuffled(g, n, torch.float32)
    elif op == "dsgesv":
        a = _shuffled(g, n, torch.float64)
    else:
        a = _randn(g, n, n)
    return a, _randn(g, case["nrhs"], n, dtype=a.dtype)


def _ivec(n):
    return torch.zeros(n, dtype=torch.int32, device=DEV)


def _ptrs(t, offsets):
    return torch.from_numpy(t.data_ptr() + t.element_size() * np.asarray(offsets, dtype=np.int64)).to(DEV)


def prepare(case, seed):
    op = case["op"]
    s = {"case": case}
    if op == "batch":
        ns, nrhs, aoff, boff, a, b = _batch_data(case, seed)
        poff = np.concatenate([[0], np.cumsum(ns)])
        s.update(a0=a, b0=b, a=torch.empty_like(a), b=torch.empty_like(b), ipiv=_ivec(int(poff[-1])),
                 info=_ivec(len(ns)), plan=la.BatchPlan(ns.tolist(), case["prec"]))
        s.update(aptr=_ptrs(s["a"], aoff[:-1]), bptr=_ptrs(s["b"], boff[:-1]), pptr=_ptrs(s["ipiv"], poff[:-1]),
                 ld=torch.from_numpy(ns.astype(np.int32)).to(DEV), nrhs=torch.from_numpy(nrhs.astype(np.int32)).to(DEV))
        return s
    if op == "adjoint":
        nb, n, r = case["batch"], case["n"], case["nrhs"]
        lu, x, xbar = _adjoint_data(case, seed)
        s.update(lu=lu, x=x, xbar=xbar, bbar=torch.empty_like(xbar), abar=torch.empty_like(lu), ipiv=_ivec(nb * n),
                 info=_ivec(nb), plan=la.BatchPlan([n] * nb, "d"))
        mat, vec = [k * n * n for k in range(nb)], [k * n * r for k in range(nb)]
        s.update(pl=_ptrs(lu, mat), px=_ptrs(x, vec), pb=_ptrs(s["bbar"], vec), pa=_ptrs(s["abar"], mat),
                 pp=_ptrs(s["ipiv"], [k * n for k in range(nb)]), ld=_ivec(nb) + n, nr=_ivec(nb) + r)
        # the forward pass, whose factors and solutions the backward pass reads
        st = torch.cuda.current_stream()
        assert s["plan"].getrf(s["pl"], s["ld"], s["pp"], s["info"], st) == 0
        assert s["plan"].getrs(s["nr"], s["pl"], s["ld"], s["pp"], s["px"], s["ld"], st) == 0
        return s
    data = _data(case, seed)
    n = case["n"]
    if op == "gesv_host":
        a, b = (t.cpu().numpy() for t in data)
        s.update(a0=a, b0=b, a=a.copy(), b=b.copy(), ipiv=np.zeros(n, np.int32))
        return s
    s.update(a0=data[0], a=torch.empty_like(data[0]), ipiv=_ivec(min(case.get("m", n), n)), info=_ivec(1))
    if op == "getrf":
        return s
    s.update(b0=data[1], b=torch.empty_like(data[1]))
    if op == "getrs":
        s["a"].copy_(s["a0"])
        assert la.dgetrf_async(n, n, s["a"], n, s["ipiv"], s["info"], torch.cuda.current_stream()) == 0
        del s["a0"]
    if op == "gesv":
        torch.cuda.synchronize()
    return s


# ---- one pass -----------------------------------------------------------------

def _ok(rc):
    if rc != 0:
        raise RuntimeError(f"the call returned {rc}")


def run(s):
    case = s["case"]
    op, n = case["op"], case.get("n")
    if op == "gesv_host":
        np.copyto(s["a"], s["a0"])
        np.copyto(s["b"], s["b0"])
        _ok(la.dgesv(n, case["nrhs"], s["a"], n, s["ipiv"], s["b"], n))
        return {"lu": s["a"], "ipiv": s["ipiv"], "x": s["b"]}
    st = torch.cuda.current_stream()
    if op == "batch":
        s["a"].copy_(s["a0"])
        s["b"].copy_(s["b0"])
        _ok(s["plan"].getrf(s["aptr"], s["ld"], s["pptr"], s["info"], st))
        _ok(s["plan"].getrs(s["nrhs"], s["aptr"], s["ld"], s["pptr"], s["bptr"], s["ld"], st))
        return {"lu": s["a"], "ipiv": s["ipiv"], "info": s["info"], "x": s["b"]}
    if op == "adjoint":
        s["bbar"].copy_(s["xbar"])
        _ok(s["plan"].adjoint(s["nr"], s["pl"], s["ld"], s["pp"], s["px"], s["ld"], s["pb"], s["ld"], s["pa"],
                              s["ld"], False, st))
        return {"abar": s["abar"], "bbar": s["bbar"]}
    if op == "getrs":
        s["b"].copy_(s["b0"])
        _ok(la.dgetrs_async(case["trans"], n, case["nrhs"], s["a"], n, s["ipiv"], s["b"], n, st))
        return {"x": s["b"]}
    if op == "getrf":
        s["a"].copy_(s["a0"])
        _ok(la.dgetrf_async(case["m"], n, s["a"], case["lda"], s["ipiv"], s["info"], st))
        return {"lu": s["a"], "ipiv": s["ipiv"], "info": s["info"]}
    if op == "dsgesv":
        # A and B are read only (A is overwritten only by the FP64 fallback)
        st.synchronize()  # the call runs on the library's own stream
        info, it = la.dsgesv(n, case["nrhs"], s["a0"], n, s["ipiv"], s["b0"], n, s["b"], n)
        _ok(info)
        return {"x": s["b"], "ipiv": s["ipiv"], "iter": it}
    s["a"].copy_(s["a0"])
    s["b"].copy_(s["b0"])
    if op == "gesv":
        st.synchronize()  # the call runs on the library's own stream
        _ok(la.dgesv(n, case["nrhs"], s["a"], n, s["ipiv"], s["b"], n))
        return {"lu": s["a"], "ipiv": s["ipiv"], "x": s["b"]}
    f, g = (la.sgetrf_async, la.sgetrs_async) if op == "lu_f32" else (la.dgetrf_async, la.dgetrs_async)
    _ok(f(n, n, s["a"], n, s["ipiv"], s["info"], st))
    _ok(g("N", n, case["nrhs"], s["a"], n, s["ipiv"], s["b"], n, st))
    return {"lu": s["a"], "ipiv": s["ipiv"], "info": s["info"], "x": s["b"]}


# ---- what a pass cannot do without ----------------------------------------------

def _lu_flops(m, n):
    k = min(m, n)
    return 2.0 * (m * n * k - (m + n) * k * k / 2.0 + k ** 3 / 3.0)


def work(case):
    op = case["op"]
    if op == "batch":
        ns, nrhs = (v.astype(np.float64) for v in _batch_sizes(case)[:2])
        es = 8 if case["prec"] == "d" else 4
        return {"bytes": es * float((2 * ns ** 2 + 2 * ns * nrhs).sum()),
                "flops": float((2.0 / 3.0 * ns ** 3 + 2 * ns ** 2 * nrhs).sum())}
    n, r = case["n"], case.get("nrhs", 0)
    if op == "adjoint":
        return {"bytes": case["batch"] * 8.0 * (2 * n * n + 4 * n * r), "flops": case["batch"] * 4.0 * n * n * r}
    if op == "getrs":
        return {"bytes": 8.0 * n * n + 16.0 * n * r, "flops": 2.0 * n * n * r}
    if op == "getrf":
        return {"bytes": 16.0 * case["m"] * n, "flops": _lu_flops(case["m"], n)}
    if op == "dsgesv":
        return {"bytes": 8.0 * n * n + 16.0 * n * r, "flops": _lu_flops(n, n) + 2.0 * n * n * r}
    es = 4.0 if op == "lu_f32" else 8.0
    return {"bytes": es * (2 * n * n + 2 * n * r), "flops": _lu_flops(n, n) + 2.0 * n * n * r}


# ---- the same results from torch in 64 bits -----------------------------------------

def _exact_lu(a, b=None):
    """Packed LU factors of the column-major matrix in a, and the solution for b, column-major (on the host)."""
    lu, p = torch.linalg.lu_factor(a.cpu().double().t())
    if b is None:
        return lu.t().contiguous()
    return lu.t().contiguous(), torch.linalg.lu_solve(lu, p, b.cpu().double().t()).t().contiguous()


def exact(case, seed):
    op = case["op"]
    if op == "batch":
        if case["batch"] * case["hi"] > 1000000:
            return None  # minutes of single factorizations
        ns, nrhs, aoff, boff, a, b = _batch_data(case, seed)
        a, b = a.cpu().double(), b.cpu().double()
        for n, r, i, j in zip(ns.tolist(), nrhs.tolist(), aoff.tolist(), boff.tolist()):
            m, v = a[i:i + n * n].view(n, n), b[j:j + n * r].view(r, n)
            lu, p = torch.linalg.lu_factor(m.t())
            v.copy_(torch.linalg.lu_solve(lu, p, v.t().contiguous()).t())
            m.copy_(lu.t())
        return {"lu": a, "ipiv": None, "info": None, "x": b}
    if op == "adjoint":
        a, b, xbar = (t.cpu() for t in _adjoint_data(case, seed))
        abar, bbar = torch.empty_like(a), torch.empty_like(xbar)
        for k in range(case["batch"]):  # a[k] holds A(i, j) at [j, i], b[k] and xbar[k] their columns as rows
            lu, p = torch.linalg.lu_factor(a[k].t())
            x = torch.linalg.lu_solve(lu, p, b[k].t().contiguous())
            bbar[k] = torch.linalg.lu_solve(lu, p, xbar[k].t().contiguous(), adjoint=True).t()
            abar[k] = -(x @ bbar[k])
        return {"abar": abar, "bbar": bbar}
    data = _data(case, seed)
    if op == "getrf":
        t = data[0].cpu()
        t[:, :case["m"]] = _exact_lu(t[:, :case["m"]].contiguous())
        return {"lu": t, "ipiv": None, "info": None}
    a, b = data
    if op == "getrs":
        return {"x": _exact_lu(a.t() if case["trans"] == "T" else a, b)[1]}
    lu, x = _exact_lu(a, b)
    if op == "dsgesv":
        return {"x": x, "ipiv": None, "iter": None}
    if op in ("gesv", "gesv_host"):
        return {"lu": lu, "ipiv": None, "x": x}
    return {"lu": lu, "ipiv": None, "info": None, "x": x}
