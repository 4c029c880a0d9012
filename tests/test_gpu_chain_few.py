"""The solve kernels by number of right-hand sides: vector sums in chunks up
to eight columns, 16-column MFMA tiles beyond, the chunks side by side. Dense
fronts around the edges of the 128-row blocks (the chained launch) and of the
16 .. 128 rows that threads are dealt by (the small fronts), and grids, whose
fronts have children and contribution blocks."""
import numpy as np
import pytest

from sylver_amd import matrices as M

pytestmark = pytest.mark.gpu

NRHS = [1, 2, 3, 8, 9, 33]


def _solver(S, A, prec):
    S.set_ext_options(precision=S.PREC_FP64 if prec == "fp64" else S.PREC_FP32, small_front_max=48,
                      refine=S.REFINE_NONE)
    opts = S.default_options()
    opts.scaling = 0
    d = S.SpLDLT(A, options=opts)
    assert d.factorize(posdef=True).flag == 0
    return d


@pytest.mark.parametrize("prec,u", [("fp64", 2.0 ** -53), ("fp32", 2.0 ** -24)])
@pytest.mark.parametrize("n", [1, 15, 17, 32, 33, 65, 127, 128, 129, 255, 256, 257, 400])
def test_dense_front_all_widths(S, O, gpu, n, prec, u):
    """n I + U[-1, 1] (condition below 2): the factorization is wrong by at
    most (n + 1) u |L| |L^T|, each triangular solve by n u |L|, so 8 n u
    bounds the error of x against the FP64 solution with room for the norms."""
    rng = np.random.default_rng(n)
    a = np.tril(rng.uniform(-1.0, 1.0, (n, n)), -1)
    a = a + a.T + n * np.eye(n)
    cols, rows = np.nonzero(np.triu(np.ones((n, n), bool)))
    d = _solver(S, M._from_coo_lower(n, rows, cols, a[rows, cols]), prec)
    x = np.asfortranarray(rng.uniform(-1.0, 1.0, (n, max(NRHS))))
    b = a @ x
    for k in NRHS:
        y = b[:, :k].copy(order="F")
        assert S.spldlt_solve(y, d.akeep, d.fkeep, options=d.options).flag == 0
        err = np.abs(y - x[:, :k]).max(axis=0) / np.abs(x[:, :k]).max(axis=0)
        assert err.max() <= 8 * n * u, (k, err)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_grid_columns_alike(S, O, gpu, prec):
    """A column's solution does not depend on the columns beside it: within a
    kernel it is the same sums (bitwise equal from chunks of the same width);
    between kernels only roundings differ. FP64: the bar of the other FP64
    solves. FP32 factors: backward errors of one size (a factor of 8)."""
    A = M.laplacian_3d(24)
    d = _solver(S, A, prec)
    b = M.random_rhs(A.n, max(NRHS), seed=5)
    sol = {}
    for k in NRHS:
        y = b[:, :k].copy(order="F")
        assert S.spldlt_solve(y, d.akeep, d.fkeep, options=d.options).flag == 0
        sol[k] = y
    assert np.array_equal(sol[3][:, :2], sol[2]) and np.array_equal(sol[8][:, :3], sol[3])
    assert np.array_equal(sol[33][:, :9], sol[9])
    errs = [O.bwd_err(A, sol[k], np.asfortranarray(b[:, :k])) for k in NRHS]
    if prec == "fp64":
        assert max(errs) <= 1e-14, errs
    else:
        assert max(errs) <= 8 * min(errs), errs


@pytest.mark.parametrize("nx,ny,nz", [(31, 17, 1), (64, 61, 1), (9, 8, 7)])
def test_ragged_small_fronts(S, O, gpu, nx, ny, nz):
    """Small fronts of many shapes (odd pivot counts, so that the rows below
    them start off 16 bytes), FP64: the bar of the other FP64 solves."""
    rng = np.random.default_rng(nx)
    g = np.arange(nx * ny * nz).reshape(nz, ny, nx)
    pairs = [(g[:, :, :-1], g[:, :, 1:]), (g[:, :-1], g[:, 1:]), (g[:-1], g[1:])]
    lo = np.concatenate([p.ravel() for p, _ in pairs] + [g.ravel()])
    hi = np.concatenate([p.ravel() for _, p in pairs] + [g.ravel()])
    val = np.where(lo == hi, 7.0, -rng.uniform(0.5, 1.0, len(lo)))
    order = np.lexsort((hi, lo))
    A = M._from_coo_lower(g.size, hi[order], lo[order], val[order])
    d = _solver(S, A, "fp64")
    b = M.random_rhs(A.n, max(NRHS), seed=6)
    for k in NRHS:
        y = b[:, :k].copy(order="F")
        assert S.spldlt_solve(y, d.akeep, d.fkeep, options=d.options).flag == 0
        assert O.bwd_err(A, y, np.asfortranarray(b[:, :k])) <= 1e-14, k
