"""The dense front LU at the edges of its size classes (one wave, four waves,
two rows a lane), on entries from {-2, -1, 1, 2}: the pivot searches meet
ties, which go to the row in the smaller position. Bit for bit the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["pp", "tpp"])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_lu_class_edges_with_ties(S, O, gpu, dtype, mode):
    rng = np.random.default_rng(4)
    m = np.array([1, 2, 16, 31, 32, 33, 63, 64, 65, 96, 127, 128, 33, 65, 128], np.int32)
    k = m.copy()
    k[-3:] = [20, 64, 1]
    off = np.zeros(len(m) + 1, np.int64)
    np.cumsum(m.astype(np.int64) ** 2, out=off[1:])
    host = rng.choice([-2.0, -1.0, 1.0, 2.0], int(off[-1])).astype(dtype)
    arr = S.DeviceArray(host)
    rc, nelim, perms = S.batched_front_lu(arr, m, k, off[:-1], dtype, mode, 0.01)
    assert rc == 0
    out = arr.numpy()
    for f in range(len(m)):
        a = host[off[f]:off[f + 1]].reshape((m[f], m[f]), order="F")
        ne, rp, cp, ref = O.lu_front(a, int(k[f]), mode, 0.01)
        got = out[off[f]:off[f + 1]].reshape((m[f], m[f]), order="F")
        assert nelim[f] == ne, m[f]
        assert np.array_equal(perms[f][0], rp) and np.array_equal(perms[f][1], cp), m[f]
        assert np.asfortranarray(got).tobytes("F") == np.asfortranarray(ref).tobytes("F"), m[f]
