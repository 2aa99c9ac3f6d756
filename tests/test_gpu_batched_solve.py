"""The batch's triangular solves (SRC/dgetrs.f:181-218) at the edges of their
blocks of 64 rows, sub-blocks of 16 and passes of 4 or 8 right-hand sides, in
each of the two workgroup sizes, against the oracle's DGETRS on the same
factors.

Tolerance: the matrices are random rows plus 4 sqrt(n) on the diagonal, their
rows shuffled, so that |L||U| stays a small multiple of |A| and the condition
number a small constant; both solutions are then within a small multiple of
n eps of the exact one (Higham, Accuracy and Stability, thm 9.4), taken as
64 n eps.  Where a result is not finite the reference's zero tests decide, and
infinities and NaNs have to be in the same places.
"""
import numpy as np
import pytest
import torch

import lapack_amd as la
import oracle

pytestmark = pytest.mark.gpu

EDGES = [1, 2, 15, 16, 17, 31, 33, 63, 64, 65, 79, 80, 81, 127, 128, 129, 191, 193, 256, 300, 513]


def factors(n, dtype, seed):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((n, n)) + 4.0 * np.sqrt(n) * np.eye(n)
    a = np.asfortranarray(a[rng.permutation(n)].astype(dtype))
    return (oracle.dgetrf if dtype == np.float64 else oracle.sgetrf)(a)[:2]


def solve(lus, pivs, rhs, trans, dtype, pad=3):
    """The batch's solve of every (lu, piv, b); lda and ldb are n + pad."""
    tdt = torch.float64 if dtype == np.float64 else torch.float32
    ns = [l.shape[0] for l in lus]
    keep, at = {}, []

    def up(m, key):
        if key not in keep:
            buf = np.full((m.shape[1] + 1, m.shape[0] + pad), 55.0, dtype=dtype)
            buf[:m.shape[1], :m.shape[0]] = m.T
            keep[key] = torch.from_numpy(buf).cuda()
        return keep[key]

    pa = [up(l, ("a", id(l))).data_ptr() for l in lus]
    pb = [up(b, ("b", k)).data_ptr() for k, b in enumerate(rhs)]
    for p in pivs:
        if ("p", id(p)) not in keep:
            keep[("p", id(p))] = torch.from_numpy(np.asarray(p, dtype=np.int32)).cuda()
    pp = [keep[("p", id(p))].data_ptr() for p in pivs]
    dev = lambda v, t: torch.tensor(v, dtype=t, device="cuda")
    pa, pb, pp = (dev(v, torch.int64) for v in (pa, pb, pp))
    ld = dev([n + pad for n in ns], torch.int32)
    nr = dev([b.shape[1] for b in rhs], torch.int32)
    plan = la.BatchPlan(ns, "d" if dtype == np.float64 else "s", autotune=False)
    if trans == "N":
        assert plan.getrs(nr, pa, ld, pp, pb, ld) == 0
    else:  # the adjoint: its first half is the transposed solve in place; X = 0, Abar = 0
        zeros = torch.zeros(max(n * max(n, b.shape[1]) for n, b in zip(ns, rhs)), dtype=tdt, device="cuda")
        outs = torch.zeros(sum(n * n for n in ns), dtype=tdt, device="cuda")
        off = np.concatenate([[0], np.cumsum([n * n for n in ns])])
        pz = dev([zeros.data_ptr()] * len(ns), torch.int64)
        po = dev([outs.data_ptr() + outs.element_size() * int(o) for o in off[:-1]], torch.int64)
        n0 = dev(ns, torch.int32)
        assert plan.adjoint(nr, pa, ld, pp, pz, n0, pb, ld, po, n0) == 0
    torch.cuda.synchronize()
    for k, (n, b) in enumerate(zip(ns, rhs)):
        buf = keep[("b", k)].cpu().numpy()
        assert (buf[:, n:] == 55.0).all() and (buf[b.shape[1]:] == 55.0).all()
        at.append(buf[:b.shape[1], :n].T)
    return at


def by_columns(lu, p, b, trans):
    """DGETRS with DTRSM's loops (BLAS/SRC/dtrsm.f:277-300, 337-362): without
    transposition a zero of the solution is not multiplied (the oracle's
    products have no such test)."""
    n, x = len(lu), b.copy()
    with np.errstate(all="ignore"):
        if trans == "N":
            for k in range(n):
                x[[k, p[k] - 1]] = x[[p[k] - 1, k]]
            for k in range(n):
                for j in np.flatnonzero(x[k] != 0):
                    x[k + 1:, j] -= x[k, j] * lu[k + 1:, k]
            for k in range(n - 1, -1, -1):
                for j in np.flatnonzero(x[k] != 0):
                    x[k, j] /= lu[k, k]
                    if x[k, j] != 0:
                        x[:k, j] -= x[k, j] * lu[:k, k]
        else:
            for k in range(n):
                x[k] = (x[k] - lu[:k, k] @ x[:k]) / lu[k, k]
            for k in range(n - 1, -1, -1):
                x[k] -= lu[k + 1:, k] @ x[k + 1:]
            for k in range(n - 1, -1, -1):
                x[[k, p[k] - 1]] = x[[p[k] - 1, k]]
    return x


def check(x, lu, p, b, trans, dtype, what):
    if np.isfinite(x).all():
        ref = (oracle.dgetrs if dtype == np.float64 else oracle.sgetrs)(lu, p, np.asfortranarray(b), trans)[0]
    else:
        ref = by_columns(lu, p, b, trans)
    tol = 64 * len(lu) * (2.0 ** -53 if dtype == np.float64 else 2.0 ** -24)
    if b.shape[1]:
        np.testing.assert_array_equal(np.isnan(x), np.isnan(ref), err_msg=what)
        np.testing.assert_array_equal(np.isinf(x) * np.sign(x), np.isinf(ref) * np.sign(ref), err_msg=what)
        fin = np.isfinite(ref)
        err = np.abs(np.where(fin, x, 0) - np.where(fin, ref, 0)).max()
        assert err <= tol * max(np.abs(ref[fin]).max(initial=0.0), 1e-30), (what, err)


@pytest.mark.parametrize("trans,dtype", [("N", np.float64), ("N", np.float32), ("T", np.float64)])
@pytest.mark.parametrize("copies", [1, 50])  # 50: more large orders than two workgroups a CU
def test_solves(dev, copies, trans, dtype):
    orders = EDGES if copies == 1 else [n for n in EDGES if n < 200]
    fs = [factors(n, dtype, 100 + n) for n in orders]
    rng = np.random.default_rng(5)
    items = [(f, rng.standard_normal((len(f[0]), r)).astype(dtype))
             for c in range(copies) for k, f in enumerate(fs) for r in [(3 * k + c) % 10 if c % 7 or copies == 1 else 17]]
    xs = solve([f[0] for f, _ in items], [f[1] for f, _ in items], [b for _, b in items], trans, dtype)
    for x, (f, b) in zip(xs, items):
        check(x, f[0], f[1], b, trans, dtype, (len(f[0]), b.shape[1]))


@pytest.mark.parametrize("trans,dtype", [("N", np.float64), ("N", np.float32), ("T", np.float64)])
def test_not_finite(dev, trans, dtype):
    """Zero, infinite and tiny diagonals, infinities off the diagonal that meet
    a zero of the solution, and overflow."""
    tiny, big = float(np.finfo(dtype).tiny) / 4, float(np.finfo(dtype).max)
    items = []
    for n in (5, 64, 130, 300):
        lu0, p = factors(n, dtype, 7 + n)
        b = np.random.default_rng(n).standard_normal((n, 3)).astype(dtype)
        for kind in ("zero_diag", "inf_diag", "tiny_diag", "inf_below", "nan_above", "overflow"):
            lu, bb = lu0.copy(order="F"), b.copy()
            if kind == "zero_diag":
                lu[n // 2, n // 2] = 0
            elif kind == "inf_diag":
                lu[n // 2, n // 2] = np.inf
            elif kind == "tiny_diag":
                lu[n - 1, n - 1] = tiny
                bb *= tiny
            elif kind == "inf_below":
                lu[n - 1, 0] = np.inf
                bb[:, 1] = 0
            elif kind == "nan_above":
                lu[0, n - 1] = np.nan
                bb[:, 1] = 0
            else:
                lu[0, 0] = 1e-3
                bb[:] = big
            items.append((lu, p, bb, kind))
    xs = solve([i[0] for i in items], [i[1] for i in items], [i[2] for i in items], trans, dtype)
    for x, (lu, p, b, kind) in zip(xs, items):
        if kind == "tiny_diag":  # gradual underflow: only that it stays finite where the oracle's is
            ref = (oracle.dgetrs if dtype == np.float64 else oracle.sgetrs)(lu, p, np.asfortranarray(b), trans)[0]
            np.testing.assert_array_equal(np.isfinite(x), np.isfinite(ref), err_msg=kind)
        elif kind == "overflow":  # which sums pass the largest number depends on their order
            ref = (oracle.dgetrs if dtype == np.float64 else oracle.sgetrs)(lu, p, np.asfortranarray(b), trans)[0]
            assert not np.isfinite(ref).all() and not np.isfinite(x).all()
        else:
            check(x, lu, p, b, trans, dtype, (len(lu), kind))


def less(x, u, v):
    """x - u v^T, every element a fused multiply-add (rounded through the next wider type)."""
    wide = np.longdouble if x.dtype != np.float32 else np.float64
    return (x.astype(wide) - np.outer(u.astype(wide), v.astype(wide))).astype(x.dtype)


def lane_sums(lu, x, trans, kb, n):
    """Sums of products of the solved rows with 64 rows' coefficients: 64 partial
    sums of every 64th product, added in a tree (rounded through 80 bits)."""
    wide = np.longdouble
    lo, hi = (0, kb) if trans == "U^T" else (min(kb + 64, n), n)
    acc = np.zeros((64, min(64, n - kb), x.shape[1]))
    for k0 in range(lo, hi, 64):
        k1 = min(k0 + 64, hi)
        u = lu[k0:k1, kb:kb + 64].astype(wide)
        acc[:k1 - k0] = (u[:, :, None] * x[k0:k1, None, :].astype(wide) + acc[:k1 - k0]).astype(np.float64)
    while len(acc) > 1:
        acc = acc[:len(acc) // 2] + acc[len(acc) // 2:]
    return acc[0]


def by_lanes(lu, b):
    """U^T then L^T, blocks of 64 rows: lane_sums, then the substitution."""
    n, x = len(lu), b.copy()
    for kb in range(0, n, 64):
        e = min(kb + 64, n)
        x[kb:e] -= lane_sums(lu, x, "U^T", kb, n)
        for k in range(kb, e):
            x[k] /= lu[k, k]
            x[k + 1:e] = less(x[k + 1:e], lu[k, k + 1:e], x[k])
    for kb in range((n - 1) // 64 * 64, -1, -64):
        e = min(kb + 64, n)
        x[kb:e] -= lane_sums(lu, x, "L^T", kb, n)
        for k in range(e - 1, kb - 1, -1):
            x[kb:k] = less(x[kb:k], lu[k, kb:k], x[k])
    return x


@pytest.mark.parametrize("copies,n,seeds", [(1, 960, 10), (600, 500, 16)])  # 16 waves; 4 waves
def test_error_of_the_transposed_solve(dev, copies, n, seeds):
    """Against 80 bits on factors of N(0,1) matrices, whose sums do not hinge on
    the diagonal: as near as with every row's product in 64 partial sums.  The
    geometric mean of the ratio over the seeds (8 right-hand sides each) may be
    1.15: its standard error is 5 to 6 %, and emulated the mean is 0.75 to 1.0."""
    logs = []
    for seed in range(seeds):
        rng = np.random.default_rng(1000 + seed)
        a = rng.standard_normal((n, n))
        lu, p = oracle.dgetrf(np.asfortranarray(a))[:2]
        b = rng.standard_normal((n, 8))
        x = solve([lu] * copies, [p] * copies, [b] * copies, "T", np.float64, pad=0)[copies // 2]
        wide, y = lu.astype(np.longdouble), b.astype(np.longdouble)
        for k in range(n):
            y[k] /= wide[k, k]
            y[k + 1:] -= np.outer(wide[k, k + 1:], y[k])
        for k in range(n - 1, -1, -1):
            y[:k] -= np.outer(wide[k, :k], y[k])
        ref = by_lanes(lu, b)
        for k in range(n - 1, -1, -1):  # the interchanges, in reverse order
            for v in (y, ref):
                v[[k, p[k] - 1]] = v[[p[k] - 1, k]]

        def err(v):
            return np.sqrt(((v - y) ** 2).sum(0).astype(float))
        logs.append(np.mean(np.log(err(x) / err(ref))))
    assert np.exp(np.mean(logs)) <= 1.15


def by_rows(lu, p, b):
    """DGETRS('N') with every row's products taken off one after the other."""
    n, x = len(lu), b.copy()
    for k in range(n):
        x[[k, p[k] - 1]] = x[[p[k] - 1, k]]
    for k in range(n):
        x[k + 1:] = less(x[k + 1:], lu[k + 1:, k], x[k])
    for k in range(n - 1, -1, -1):
        x[k] /= lu[k, k]
        x[:k] = less(x[:k], lu[:k, k], x[k])
    return x


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_error_of_the_solve(dev, dtype):
    """The same for DGETRS('N') in 4 waves, against the order of DTRSM's loops."""
    n, copies, logs = 500, 600, []
    wide = np.longdouble if dtype == np.float64 else np.float64
    for seed in range(16):
        rng = np.random.default_rng(2000 + seed)
        lu, p = oracle.dgetrf(np.asfortranarray(rng.standard_normal((n, n))))[:2]
        lu = np.asfortranarray(lu.astype(dtype))
        b = rng.standard_normal((n, 8)).astype(dtype)
        x = solve([lu] * copies, [p] * copies, [b] * copies, "N", dtype, pad=0)[copies // 2]
        y, ref = by_rows(lu.astype(wide), p, b.astype(wide)), by_rows(lu, p, b)

        def err(v):
            return np.sqrt(((v - y) ** 2).sum(0).astype(float))
        logs.append(np.mean(np.log(err(x) / err(ref))))
    assert np.exp(np.mean(logs)) <= 1.1
