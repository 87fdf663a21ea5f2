"""Zero pivots are reported by every line solver (csrc/diffuse.hip): a first
row whose diagonal cancels to zero, without off-diagonal entries, is a
dominant M-matrix row by its factors' signs, so the sweep stays with the
partitioned solves, and the factorisation that finds the pivot has to run all
the same."""
import numpy as np
import pytest

from test_gpu_parity import assert_same, tr  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dirn", ["x", "y", "z"])
@pytest.mark.parametrize("solver", ["partitioned", "exact"])
def test_zero_pivot_without_off_diagonals(pkg, oracle, tr, dirn, solver):  # noqa: F811
    st = pkg.workloads.random_state(12, 9, 11, 2, seed=3, latlon=True)
    q = st.concen_pd.copy()
    k = np.moveaxis(getattr(st, "k" + dirn), "xyz".index(dirn), 0)
    was = k.copy()
    T = tr.Transport(st)
    T.tune(line_solver=solver)
    # L = 1e40-like, R = 0: 1 + th*(L + R) - th*L is zero
    k[0, 3, 4], k[1, 3, 4], k[2, 3, 4] = 1.0e40, 0.0, 0.0
    T.sync_from_host(tr.SYNC_DIFFK)
    getattr(T, "diffCN_" + dirn)()
    with pytest.raises(tr.Ash3dError, match="zero pivot"):
        T.synchronize()
    # and no more once the line is regular again
    k[...] = was
    st.concen_pd[...] = q
    T.sync_from_host(tr.SYNC_DIFFK | tr.SYNC_CONCEN)
    a = st.copy()
    getattr(T, "diffCN_" + dirn)()
    O = oracle.Oracle(a)
    getattr(O, "diffCN_" + dirn)()
    T.sync_to_host()
    assert_same(a, st, tol=0.0 if solver == "exact" else 1e-12)
    T.close()
