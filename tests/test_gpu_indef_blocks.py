"""Pivoting of the indefinite panels at the edges of their 64-column blocks
and 64-row groups, on entries from {-2, -1, 1, 2} with half the diagonal zero:
the largest entry of a block is met many times over (the first by column, then
row, is the pivot) and 2 x 2 pivots are common. Both panels, bit for bit the
oracle's front."""
import numpy as np
import pytest

from test_gpu_indef_fronts import SMALL, U, _front_tree, _seam_factor, _seam_free

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("panel_min", [1, 10000])
@pytest.mark.parametrize("m,n", [(1, 1), (2, 2), (17, 17), (63, 63), (64, 64), (65, 65), (129, 64), (130, 65),
                                 (200, 100), (330, 70)])
def test_block_edges_with_ties(S, O, gpu, m, n, panel_min):
    rng = np.random.default_rng(100 * m + n)
    a = np.tril(rng.choice([-2.0, -1.0, 1.0, 2.0], (m, m)))
    if m > 1:
        half = rng.permutation(m)[:m // 2]
        a[half, half] = 0.0
    a = a + np.tril(a, -1).T
    A, sym = _front_tree(S, O, a, m, n)
    S.set_ext_options(precision=S.PREC_FP64, indef_panel_min=panel_min)
    L, tree, nt, ic = _seam_factor(S, A, sym)
    try:
        assert nt and ic.flag == 0, ic.flag
        ref = O.IndefFactor(sym, A.val, nb=64, u=U, small=SMALL)
        got, want = S.fkeep_indef_node(nt, 0), ref.node(0)
        assert got["nelim"] == want["nelim"]
        assert np.array_equal(got["rows"], want["rows"])
        assert np.array_equal(got["dinv"], want["dinv"])
        assert np.array_equal(np.tril(got["L"], -1), np.tril(want["L"], -1))
        assert (ic.num_delay, ic.num_two, ic.num_neg) == tuple(
            ref.stats[k] for k in ("num_delay", "num_two", "num_neg"))
    finally:
        S.set_ext_options(indef_panel_min=0)
        _seam_free(S, L, tree, nt)
