"""dgtsv-order solves of a box or of few bins (csrc/cn_exact.hip): workgroups
(64 lines by four, two or one bins) without a line of the box or an aloft bin
store zeros only.  Bitwise the oracle, on lines that run in registers (64 and
80 cells) and through the ts1 slot."""
import numpy as np
import pytest

from test_gpu_parity import assert_same, run_both, tr  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mask", [(1,) * 9, (0, 0, 0, 0, 1, 0, 1, 0, 0), (0,) * 8 + (1,), (0,) * 9, (0, 1, 0), (0, 0, 1),
                                  (0, 1), (1,), (0,)])
@pytest.mark.parametrize("shape,box", [((70, 66, 9), (30, 36, 12, 14, 4, 6)), ((70, 66, 9), (1, 3, 64, 66, 7, 9)),
                                       ((7, 131, 70), (2, 5, 100, 131, 1, 70)), ((131, 5, 85), (1, 131, 1, 5, 3, 85)),
                                       ((131, 5, 85), (70, 80, 3, 5, 1, 3))])
def test_boxes(pkg, oracle, tr, shape, box, mask):  # noqa: F811
    st = pkg.workloads.random_state(*shape, len(mask), seed=sum(box) + len(mask), latlon=True)
    st.bounds = box
    st.is_aloft = np.array(mask, dtype=np.int32)
    calls = [("diffCN_x",), ("diffCN_y",), ("diffCN_z",)]
    a, b = run_both(pkg, oracle, tr, st, calls + calls)
    assert_same(a, b)
