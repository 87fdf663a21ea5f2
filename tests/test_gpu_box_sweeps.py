"""Sweeps of a small box or of few bins (csrc/advect_tile.hip): tiles with no
line or cell of the box and bins that are not aloft are stored as zeros and
not read.  Bitwise the oracle for boxes that leave out tiles of lines (64) and
of cells (5, 6 and 8 a wave, 20 a workgroup) on either side, in place and
through ts1, and cheaper than the sweep of the whole grid."""
import numpy as np
import pytest

from test_gpu_parity import assert_same, run_both, tr  # noqa: F401

pytestmark = pytest.mark.gpu

MASKS = [(1,) * 9, (1, 0, 0, 1, 1, 0, 1, 0, 0), (0,) * 8 + (1,), (0,) * 9]


@pytest.mark.parametrize("mask", MASKS)
@pytest.mark.parametrize("box", [(66, 70, 12, 14, 9, 11), (1, 3, 1, 2, 1, 3), (139, 140, 44, 45, 2, 4),
                                 (60, 130, 21, 40, 13, 26), (1, 140, 1, 45, 1, 27)])
@pytest.mark.parametrize("topo", [False, True])
def test_boxes_in_place(pkg, oracle, tr, box, mask, topo):  # noqa: F811
    st = pkg.workloads.random_state(140, 45, 27, 9, seed=sum(box), latlon=True, zscaling_id=2 if topo else 0)
    st.bounds = box
    st.is_aloft = np.array(mask, dtype=np.int32)
    a, b = run_both(pkg, oracle, tr, st, [("advect_y",), ("advect_z",), ("advect_y",)])
    assert_same(a, b)


@pytest.mark.parametrize("mask", MASKS)
@pytest.mark.parametrize("vent", [(70, 13, 5), (2, 2, 2), (139, 44, 20)])
@pytest.mark.parametrize("use_diffusion", [False, True])
def test_boxes_through_ts1(pkg, oracle, tr, vent, mask, use_diffusion):  # noqa: F811
    st = pkg.workloads.random_state(140, 45, 27, 9, seed=sum(vent), latlon=True)
    cloud = np.zeros_like(st.concen_pd)
    i, j, k = (v + 1 for v in vent)
    cloud[i - 2:i + 2, j - 2:j + 2, k - 2:k + 3] = st.concen_pd[i - 2:i + 2, j - 2:j + 2, k - 2:k + 3]
    cloud[:2], cloud[-2:], cloud[:, :2], cloud[:, -2:], cloud[:, :, :2], cloud[:, :, -2:] = (0,) * 6
    st.concen_pd = np.asfortranarray(cloud)
    st.concen_pd[..., 1] = st.concen_pd[..., 0]
    st.is_aloft = np.array(mask, dtype=np.int32)
    a, b = st.copy(), st.copy()
    O, T = oracle.Oracle(a), tr.Transport(b)
    T.tune(line_solver="exact")
    for itime in (1, 2):
        for S in (O, T):
            S.step_glue()
            S.transport_step_subgrid(itime, use_diffusion, *vent)
    T.sync_to_host()
    assert_same(a, b)
    T.close()


@pytest.mark.parametrize("kinds", ["advect"])
def test_small_boxes_cost_less(pkg, tr, kinds):  # noqa: F811
    """GPU time of the sweeps of a 3x3x3 box against the whole grid's."""
    st = pkg.workloads.random_state(240, 160, 40, 6, seed=4, latlon=True)
    T = tr.Transport(st)
    T.tune(line_solver="exact")
    best = {}
    for itime in range(1, 13):
        thresh = 1.0e30 if itime % 4 < 2 else 0.0
        T.profile(True)
        T.transport_step_subgrid(itime, True, 120, 80, 2, thresh)
        T.synchronize()
        prof = T.profile_read()
        T.profile(False)
        for kind in (kinds + "_y", kinds + "_z"):
            best[kind, thresh] = min(best.get((kind, thresh), 1.0e9), prof[kind][0])
    for kind in (kinds + "_y", kinds + "_z"):
        assert best[kind, 1.0e30] < 0.8 * best[kind, 0.0], (kind, best)
    T.close()
