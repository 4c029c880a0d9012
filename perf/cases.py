"""The workloads whose time is followed, through the package's public calls.

Four kinds of work, each over the sizes it is used at:

``factor_solve``
    One numeric factorization and one solve with an analysis (and a factor
    handle) that the program keeps: a new set of values on a known pattern,
    as in a Newton or time step. Positive definite grid operators in FP64,
    or in FP32 with the FP64 refinement inside the solve.
``solve``
    A further solve with factors that are already there.
``kkt``
    ``factor_solve`` for a saddle-point matrix: the indefinite path with
    delayed pivots.
``potrf``, ``lu``
    Many dense fronts of differing sizes factored in one call, on device
    data that the caller has just (re)assembled.

A right-hand side is made from a known solution, so that solution is what a
solve ought to return.
"""
from __future__ import annotations

import ctypes
import functools
import math
import types

import numpy as np
import torch

import sylver_amd as S
from sylver_amd import matrices as M


def listed():
    return [
        # the smallest call: a coarse-grid or sub-domain solve, all latency
        dict(name="grid3d_12_fp64", kind="factor_solve", nx=12, ny=12, nz=12, prec="fp64", nrhs=2, scaling=0),
        # a small 2D problem (n = 10,000), one right-hand side
        dict(name="grid2d_100_fp64", kind="factor_solve", nx=100, ny=100, nz=1, prec="fp64", nrhs=1, scaling=0),
        # a large, ragged 2D problem in the low-precision tier: many small fronts, a refined solve
        dict(name="grid2d_701x523_fp32", kind="factor_solve", nx=701, ny=523, nz=1, prec="fp32", nrhs=1, scaling=0),
        # an ordinary 3D problem of odd sides, equilibrated
        dict(name="grid3d_47x39x31_fp64", kind="factor_solve", nx=47, ny=39, nz=31, prec="fp64", nrhs=3, scaling=4),
        # the benchmark's configuration: 80^3, FP32 factors, 16 refined right-hand sides
        dict(name="grid3d_80_fp32_rhs16", kind="factor_solve", nx=80, ny=80, nz=80, prec="fp32", nrhs=16, scaling=0),
        # the same grid in plain FP64, one right-hand side: the largest
        dict(name="grid3d_80_fp64", kind="factor_solve", nx=80, ny=80, nz=80, prec="fp64", nrhs=1, scaling=0),
        # a step that reuses its factors, one right-hand side
        dict(name="solve_61x60x59_fp64", kind="solve", nx=61, ny=60, nz=59, prec="fp64", nrhs=1, scaling=0),
        # a block of right-hand sides (an odd number of them) against FP32 factors, refined
        dict(name="solve_53x50x47_fp32_rhs33", kind="solve", nx=53, ny=50, nz=47, prec="fp32", nrhs=33, scaling=0),
        # a saddle-point system: constrained 20^3 grid, a constraint row per four unknowns
        dict(name="kkt_20_fp64", kind="kkt", side=20, rows=2000, prec="fp64", nrhs=1),
        # dense fronts of a multifrontal code, partial Cholesky, 8 to 256 pivots each
        dict(name="potrf_4000_fp64", kind="potrf", fronts=4000, sizes=1, prec="fp64"),
        dict(name="potrf_1500_fp32", kind="potrf", fronts=1500, sizes=2, prec="fp32"),
        # dense fronts of an unsymmetric code, partial pivoting, orders 8 to 128
        dict(name="lu_pp_4000_fp64", kind="lu", fronts=4000, sizes=5, prec="fp64", mode="pp", part=1.0),
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], spread evenly over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    kind = rng.choice(["factor_solve", "factor_solve", "solve", "kkt", "potrf", "lu"])
    prec = rng.choice(["fp64", "fp32"])
    if kind in ("factor_solve", "solve"):
        if rng.random() < 0.4:
            nx = _log_int(rng, 30, 700)
            ny, nz = max(20, int(nx * rng.uniform(0.5, 1.0))), 1
        else:
            nx = _log_int(rng, 10, 72)
            ny = max(5, int(nx * rng.uniform(0.6, 1.0)))
            nz = max(4, int(nx * rng.uniform(0.4, 1.0)))
        nrhs = min(_log_int(rng, 1, 40), max(1, 4_000_000 // (nx * ny * nz)))
        scaling = rng.choice([0, 0, 4]) if kind == "factor_solve" else 0
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, prec=prec, nrhs=nrhs, scaling=scaling)
    if kind == "kkt":
        side = _log_int(rng, 6, 20)
        return dict(kind=kind, side=side, rows=max(8, int(side ** 3 * rng.uniform(0.1, 0.25))), prec=prec,
                    nrhs=_log_int(rng, 1, 8))
    case = dict(kind=kind, fronts=_log_int(rng, 30, 4000), sizes=rng.randrange(1000), prec=prec)
    if kind == "lu":
        case.update(mode=rng.choice(["pp", "tpp", "nopiv"]), part=rng.choice([1.0, round(rng.uniform(0.3, 1.0), 2)]))
    return case


# ---- sparse systems -------------------------------------------------------
def _columns(A):
    return np.repeat(np.arange(A.n, dtype=np.int64), np.diff(A.ptr))


def _grid(case, seed):
    """A grid operator with edge coefficients in [0.5, 1.5] and the Dirichlet
    boundary's ones on the diagonal: symmetric positive definite."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    A = M.laplacian_3d(nx, ny, nz, diag=6.0 if nz > 1 else 4.0)
    rng = np.random.default_rng((seed, 11))
    cols, rows = _columns(A), A.row.astype(np.int64) - 1
    off = rows != cols
    coef = rng.uniform(0.5, 1.5, int(off.sum()))
    A.val[off] = -coef
    missing = (6 if nz > 1 else 4) - np.bincount(cols[off], minlength=A.n) - np.bincount(rows[off], minlength=A.n)
    A.val[~off] = (missing + np.bincount(cols[off], coef, A.n) + np.bincount(rows[off], coef, A.n))[cols[~off]]
    return A


def _kkt(case, seed):
    """[H A^T; A 0] on a fixed pattern: the Laplacian with coefficients in
    [1, 2] added to its diagonal, constraint entries uniform in [-1, 1]."""
    K = M.kkt(case["side"], case["rows"], seed=3)
    rng = np.random.default_rng((seed, 12))
    cols, rows = _columns(K), K.row.astype(np.int64) - 1
    con = rows >= case["side"] ** 3
    K.val[con] = rng.uniform(-1.0, 1.0, int(con.sum()))
    diag = rows == cols
    K.val[diag] += rng.uniform(1.0, 2.0, int(diag.sum()))
    return K


def _solution(case, seed):
    n = case["side"] ** 3 + case["rows"] if case["kind"] == "kkt" else case["nx"] * case["ny"] * case["nz"]
    rng = np.random.default_rng((seed, 13))
    return np.asfortranarray(rng.uniform(-1.0, 1.0, size=(case["nrhs"], n)).T)


def _product(A, x):
    cols, rows = _columns(A), A.row.astype(np.int64) - 1
    low = rows != cols
    b = np.empty_like(x, order="F")
    for k in range(x.shape[1]):
        xk = x[:, k]
        b[:, k] = np.bincount(rows, A.val * xk[cols], A.n) + np.bincount(cols[low], A.val[low] * xk[rows[low]], A.n)
    return b


def _prepare_sparse(case, seed):
    A = _kkt(case, seed) if case["kind"] == "kkt" else _grid(case, seed)
    opts = S.default_options()
    opts.scaling = case.get("scaling", 0)
    st = types.SimpleNamespace(kind=case["kind"], posdef=case["kind"] != "kkt",
                               precision=S.PREC_FP64 if case["prec"] == "fp64" else S.PREC_FP32,
                               solver=S.SpLDLT(A, options=opts), b=_product(A, _solution(case, seed)))
    st.x = np.empty_like(st.b, order="F")
    if case["kind"] == "solve":
        S.set_ext_options(precision=st.precision)
        _factorize(st)
    return st


def _factorize(st):
    if st.solver.factorize(posdef=st.posdef).flag < 0:
        raise RuntimeError(f"factorization failed: flag {st.solver.factor_inform.flag}")


def _run_sparse(st):
    S.set_ext_options(precision=st.precision)
    if st.kind != "solve":
        _factorize(st)
    np.copyto(st.x, st.b)
    d = st.solver
    inform = S.spldlt_solve(st.x, d.akeep, d.fkeep, options=d.options)
    if inform.flag < 0:
        raise RuntimeError(f"solve failed: flag {inform.flag}")
    if st.kind == "kkt":
        return {"x": st.x, "num_neg": int(d.factor_inform.num_neg)}
    return {"x": st.x}


@functools.lru_cache(maxsize=64)
def _symbolic(kind, *dims):
    """Entries of the matrix, entries of the factor and factorization flops."""
    A = M.kkt(dims[0], dims[1], seed=3) if kind == "kkt" else M.laplacian_3d(*dims)
    akeep, inform, _ = S.spldlt_analyse(A.n, A.ptr, A.row, A.val)
    S.spldlt_free_akeep(akeep)
    return A.n, A.nnz, int(inform.num_factor), int(inform.num_flops)


def _work_sparse(case):
    if case["kind"] == "kkt":
        n, nnz, factor, flops = _symbolic("kkt", case["side"], case["rows"])
    else:
        n, nnz, factor, flops = _symbolic("grid", case["nx"], case["ny"], case["nz"])
    es = 8 if case["prec"] == "fp64" else 4
    # one forward and one backward sweep over the factor; x in and out
    bytes_, ops = 2 * factor * es + 16 * n * case["nrhs"], 4 * factor * case["nrhs"]
    if case["kind"] != "solve":
        bytes_, ops = bytes_ + 8 * nnz + factor * es, ops + flops
    return {"bytes": bytes_, "flops": ops}


# ---- batches of dense fronts ----------------------------------------------
def _front_sizes(case):
    if case["kind"] == "potrf":
        return M.dense_front_sizes(case["fronts"], seed=case["sizes"])
    rng = np.random.default_rng(case["sizes"])
    m = np.exp(rng.uniform(np.log(8), np.log(128.999), case["fronts"])).astype(np.int32)
    return m, np.maximum(1, (m * case["part"]).astype(np.int32))


def _front_offsets(m):
    off = np.zeros(len(m) + 1, np.int64)
    np.cumsum(m.astype(np.int64) ** 2, out=off[1:])
    return off


def _front_values(case, seed):
    """Entries uniform in [-1, 1]; the order added to the diagonal where no
    pivoting will see to it. Column-major squares one after the other."""
    m, _ = _front_sizes(case)
    off = _front_offsets(m)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = torch.float64 if case["prec"] == "fp64" else torch.float32
    v = torch.rand(int(off[-1]), dtype=dtype, device="cuda", generator=gen).mul_(2.0).sub_(1.0)
    if case["kind"] == "potrf" or case["mode"] == "nopiv":
        m64 = m.astype(np.int64)
        k = np.arange(int(m64.sum())) - np.repeat(np.cumsum(m64) - m64, m64)
        at = np.repeat(off[:-1], m64) + k * (np.repeat(m64, m64) + 1)
        v[torch.from_numpy(at).cuda()] += torch.from_numpy(np.repeat(m64, m64)).cuda().to(dtype)
    return v


def _prepare_fronts(case, seed):
    m, n = _front_sizes(case)
    assembled = _front_values(case, seed)
    fronts = torch.empty_like(assembled)
    return types.SimpleNamespace(kind=case["kind"], m=m, n=n, off=_front_offsets(m)[:-1].copy(), mode=case.get("mode"),
                                 dtype=np.float64 if case["prec"] == "fp64" else np.float32, assembled=assembled,
                                 fronts=fronts, device=types.SimpleNamespace(ptr=ctypes.c_void_p(fronts.data_ptr())))


def _run_fronts(st):
    st.fronts.copy_(st.assembled)  # the fronts are factored in place
    if st.kind == "potrf":
        rc, info, _ = S.batched_front_potrf(st.device, st.m, st.n, st.off, st.dtype)
        if rc != 0:
            raise RuntimeError(f"batched factorization failed: {rc}")
        return {"fronts": st.fronts, "info": info}
    rc, nelim, perms = S.batched_front_lu(st.device, st.m, st.n, st.off, st.dtype, st.mode)
    if rc != 0:
        raise RuntimeError(f"batched factorization failed: {rc}")
    return {"fronts": st.fronts, "nelim": nelim, "rows": np.concatenate([p[0] for p in perms]),
            "columns": np.concatenate([p[1] for p in perms])}


def _work_fronts(case):
    m, n = (a.astype(np.float64) for a in _front_sizes(case))
    es = 8 if case["prec"] == "fp64" else 4
    q = m - n
    if case["kind"] == "potrf":
        return {"bytes": float(es * (m * (m + 1)).sum()), "flops": float((n ** 3 / 3 + q * n ** 2 + q ** 2 * n).sum())}
    return {"bytes": float(2 * es * (m ** 2).sum()), "flops": float((2 * (m ** 3 - q ** 3) / 3).sum())}


def _exact_fronts(case, seed):
    if case["kind"] == "lu" and (case["mode"] == "tpp" or case["prec"] == "fp32"):
        return None  # the pivots depend on the type's own rounding
    m, n = _front_sizes(case)
    off = _front_offsets(m)
    flat = _front_values(case, seed).to("cpu", torch.float64)
    threads = torch.get_num_threads()
    torch.set_num_threads(1)
    for f in range(len(m)):
        mf, k = int(m[f]), int(n[f])
        a = flat[int(off[f]):int(off[f + 1])].view(mf, mf).T  # the column-major front
        if case["kind"] == "potrf":
            l11 = torch.linalg.cholesky(torch.tril(a[:k, :k]) + torch.tril(a[:k, :k], -1).T)
            l21 = torch.linalg.solve_triangular(l11.T, a[k:, :k], upper=True, left=False)
            low = torch.tril(torch.ones(mf, mf, dtype=torch.bool))
            a[k:, k:] -= torch.where(low[k:, k:], l21 @ l21.T, 0.0)
            a[k:, :k] = l21
            a[:k, :k] = torch.where(low[:k, :k], l11, a[:k, :k])
            continue
        order = torch.arange(mf)
        if case["mode"] == "pp":
            lu, piv = torch.linalg.lu_factor(a[:, :k].contiguous())
            for j, p in enumerate((piv - 1).tolist()):
                order[j], order[p] = order[p].clone(), order[j].clone()
        else:
            top, _ = torch.linalg.lu_factor(a[:k, :k].cuda().contiguous(), pivot=False)
            top = top.cpu()
            lu = torch.cat([top, torch.linalg.solve_triangular(torch.triu(top), a[k:, :k], upper=True, left=False)])
        right = a[:, k:][order]
        u12 = torch.linalg.solve_triangular(torch.tril(lu[:k], -1), right[:k], upper=False, unitriangular=True)
        a[:, k:] = torch.cat([u12, right[k:] - lu[k:] @ u12])
        a[:, :k] = lu
    torch.set_num_threads(threads)
    if case["kind"] == "potrf":
        return {"fronts": flat, "info": None}
    return {"fronts": flat, "nelim": None, "rows": None, "columns": None}


# ---- what the measurement calls ---------------------------------------------
def prepare(case, seed):
    return _prepare_fronts(case, seed) if case["kind"] in ("potrf", "lu") else _prepare_sparse(case, seed)


def run(state):
    return _run_fronts(state) if state.kind in ("potrf", "lu") else _run_sparse(state)


def work(case):
    return _work_fronts(case) if case["kind"] in ("potrf", "lu") else _work_sparse(case)


def exact(case, seed):
    if case["kind"] in ("potrf", "lu"):
        return _exact_fronts(case, seed)
    x = _solution(case, seed)
    return {"x": x, "num_neg": None} if case["kind"] == "kkt" else {"x": x}
