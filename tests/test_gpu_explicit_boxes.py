"""Explicit diffusion of a box or of few bins (csrc/diffuse_explicit.hip):
tiles without a line or cell of the box, and bins that are not aloft, are
stored as zeros and not read.  Bitwise the oracle, for lines of one workgroup
(64 cells) and several, and cheaper than the sweep of the whole grid."""
import numpy as np
import pytest

from test_gpu_parity import assert_same, run_both, tr  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mask", [(1,) * 9, (0, 1, 0, 0, 1, 0, 1, 1, 0), (0,) * 8 + (1,), (0,) * 9, (1, 0)])
@pytest.mark.parametrize("shape,box", [((70, 140, 9), (30, 36, 62, 66, 4, 6)), ((70, 140, 9), (1, 3, 138, 140, 7, 9)),
                                       ((131, 9, 70), (66, 131, 2, 5, 64, 70)), ((131, 9, 70), (1, 5, 3, 3, 1, 8)),
                                       ((70, 65, 65), (1, 70, 1, 65, 1, 65))])
def test_boxes(pkg, oracle, tr, shape, box, mask):  # noqa: F811
    st = pkg.workloads.random_state(*shape, len(mask), seed=sum(box) + len(mask), latlon=True, use_cn=False)
    st.dt *= 0.2
    st.bounds = box
    st.is_aloft = np.array(mask, dtype=np.int32)
    calls = [("diff_x",), ("diff_y",), ("diff_z",)]
    a, b = run_both(pkg, oracle, tr, st, calls + calls)
    assert_same(a, b)


def test_small_boxes_cost_less(pkg, tr):  # noqa: F811
    """GPU time of the sweeps of a 5x5x5 box against the whole grid's."""
    st = pkg.workloads.random_state(240, 160, 40, 6, seed=4, latlon=True, use_cn=False)
    T = tr.Transport(st)
    best = {}
    for k in range(12):
        box = (118, 122, 78, 82, 1, 5) if k % 2 else (1, 240, 1, 160, 1, 40)
        st.bounds = box
        T.profile(True)
        T.diff_y()
        T.diff_z()
        T.synchronize()
        prof = T.profile_read()
        T.profile(False)
        for kind in ("diffuse_y", "diffuse_z"):
            best[kind, k % 2] = min(best.get((kind, k % 2), 1.0e9), prof[kind][0])
    for kind in ("diffuse_y", "diffuse_z"):
        assert best[kind, 1] < 0.8 * best[kind, 0], (kind, best)
    T.close()
