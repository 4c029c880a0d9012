"""The one-workgroup front factorization (front_potrf_block) at the edges of
its blocking, against numpy in FP64: 16-column panels, 16-row strips, one or
several passes over the rows (384 rows a pass), 32 x 32 contribution tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (2, 1), (3, 0), (15, 15), (16, 16), (17, 16), (17, 17), (33, 32), (31, 7), (65, 64), (100, 37),
          (129, 128), (144, 16), (145, 17), (272, 16), (273, 20), (400, 16), (401, 17), (410, 390), (257, 100),
          (800, 40)]


def _reference(a, n):
    m = a.shape[0]
    ref = a.copy()
    if n:
        full = np.tril(a) + np.tril(a, -1).T
        l11 = np.linalg.cholesky(full[:n, :n])
        l21 = np.linalg.solve(l11, full[n:, :n].T).T
        ref[:n, :n] = np.where(np.tri(n, dtype=bool), l11, a[:n, :n])
        ref[n:, :n] = l21
        ref[n:, n:] = np.where(np.tri(m - n, dtype=bool), a[n:, n:] - l21 @ l21.T, a[n:, n:])
    return ref


def _layout(shapes):
    m = np.array([s[0] for s in shapes], np.int32)
    n = np.array([s[1] for s in shapes], np.int32)
    off = np.zeros(len(m) + 1, np.int64)
    np.cumsum(m.astype(np.int64) ** 2, out=off[1:])
    return m, n, off


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_front_block_edges(S, gpu, dtype):
    """Lower triangle within 8 n eps of the largest entry (the fronts are
    diagonally dominant, so nothing grows); the upper triangle untouched."""
    m, n, off = _layout(SHAPES)
    arr = S.DeviceArray.empty(int(off[-1]), dtype)
    assert S.batched_front_fill(arr, m, off[:-1], dtype, 7) == 0
    host = arr.numpy()
    rc, info, _ = S.batched_front_potrf(arr, m, n, off[:-1], dtype)
    assert rc == 0 and not info.any()
    out = arr.numpy()
    for f in range(len(m)):
        mf, nf = int(m[f]), int(n[f])
        a = host[off[f]:off[f + 1]].reshape(mf, mf, order="F").astype(np.float64)
        got = out[off[f]:off[f + 1]].reshape(mf, mf, order="F").astype(np.float64)
        ref = _reference(a, nf)
        tol = 8 * max(nf, 1) * np.finfo(dtype).eps * max(1.0, np.abs(ref).max())
        assert np.abs(np.tril(got - ref)).max() <= tol, (mf, nf)
        assert np.array_equal(np.triu(got, 1), np.triu(a, 1)), (mf, nf)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("column", [0, 15, 16, 37, 47])
def test_front_block_reports_pivot(S, gpu, dtype, column):
    """info is the 1-based column of the first non-positive pivot; the other
    fronts of the call are factored all the same."""
    shapes = [(60, 48), (430, 48), (60, 48)]
    m, n, off = _layout(shapes)
    host = np.zeros(int(off[-1]), dtype)
    for f, (mf, _) in enumerate(shapes):
        a = np.eye(mf) * mf
        if f < 2:
            a[column, column] = 0.0 if f else -1.0
        host[off[f]:off[f + 1]] = a.reshape(-1, order="F").astype(dtype)
    arr = S.DeviceArray(host)
    rc, info, _ = S.batched_front_potrf(arr, m, n, off[:-1], dtype)
    assert rc == 0
    assert info.tolist() == [column + 1, column + 1, 0]
    last = arr.numpy()[off[2]:].reshape(60, 60, order="F")
    assert np.allclose(np.diag(last)[:48], np.sqrt(60.0), rtol=4 * np.finfo(dtype).eps, atol=0)
