"""The streamed y and z sweeps (csrc/advect.hip) where they run: in place along
more than 64 cells, and z boxes that reach the top without starting at the
bottom; every number of bins per thread, cut lines and bin groups per
workgroup.  Bitwise the oracle."""
import numpy as np
import pytest

from test_gpu_parity import assert_same, tr  # noqa: F401

pytestmark = pytest.mark.gpu


def both(oracle, tr, st, calls, **settings):  # noqa: F811
    a, b = st.copy(), st.copy()
    O, T = oracle.Oracle(a), tr.Transport(b)
    T.tune(**settings)
    for name in calls:
        getattr(O, name)()
        getattr(T, name)()
    T.sync_to_host()
    T.close()
    assert_same(a, b)


@pytest.mark.parametrize("nb", [1, 2, 3, 4, 8])
@pytest.mark.parametrize("groups", [0, 1, 3, 4])
@pytest.mark.parametrize("topo", [False, True])
def test_long_lines(pkg, oracle, tr, nb, groups, topo):  # noqa: F811
    kw = dict(latlon=True, zscaling_id=2 if topo else 0)
    settings = dict(nb_advect_y=nb, nb_advect_z=nb, adv_groups_y=groups, adv_groups_z=groups)
    mask = np.array([1, 1, 0, 1, 1, 1, 1], dtype=np.int32)
    st = pkg.workloads.random_state(70, 67, 5, 7, seed=17 + nb, **kw)
    st.is_aloft = mask
    both(oracle, tr, st, ["advect_y", "advect_y"], **settings)
    st = pkg.workloads.random_state(70, 5, 67, 7, seed=18 + nb, **kw)
    st.is_aloft = mask
    both(oracle, tr, st, ["advect_z", "AdvectVert"], **settings)


@pytest.mark.parametrize("nb", [1, 2, 3, 8])
@pytest.mark.parametrize("groups", [0, 4])
def test_boxes_at_the_top(pkg, oracle, tr, nb, groups):  # noqa: F811
    st = pkg.workloads.random_state(70, 9, 30, 7, seed=5, latlon=True)
    st.bounds = (3, 69, 2, 8, 6, 30)
    both(oracle, tr, st, ["advect_z", "advect_z"], nb_advect_z=nb, adv_groups_z=groups)
