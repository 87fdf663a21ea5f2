"""Tiles of the partitioned line solves (csrc/linesolve.hip): strided lines at
the edges of each tile shape (16 lanes of 4, 5, 6 rows, 32 of 4 and 8), 8 or
16 lines per tile by the number of bins, line counts around a tile, lines
shorter than the lanes of a tile (the set-up reads every lane's first row),
contiguous lines around 64 lanes of 4 and 6 rows, boxes and masks; the
oracle's dgtsv-order solves to 1e-12 of the largest value, the bar of the
other tests of these solves."""
import numpy as np
import pytest

from test_gpu_parity import assert_same, tr  # noqa: F401

pytestmark = pytest.mark.gpu

TOL = 1e-12


def sweeps(pkg, oracle, tr, shape, ns, names, scale=20.0, **tune):  # noqa: F811
    st = pkg.workloads.random_state(*shape, ns, seed=sum(shape) + ns, latlon=True)
    st.dt *= scale
    a, b = st.copy(), st.copy()
    O, T = oracle.Oracle(a), tr.Transport(b)
    T.tune(line_solver="partitioned", jacobi_sweeps=0, **tune)
    for name in names:
        getattr(O, name)()
        getattr(T, name)()
    T.sync_to_host()
    T.close()
    assert_same(a, b, tol=TOL)


@pytest.mark.parametrize("n", [3, 4, 15, 16, 17, 63, 64, 65, 80, 81, 96, 97, 128, 129, 255, 256])
@pytest.mark.parametrize("ns", [1, 8, 9])
def test_strided(pkg, oracle, tr, n, ns):  # noqa: F811
    sweeps(pkg, oracle, tr, (17, n, 3), ns, ["diffCN_y"])
    sweeps(pkg, oracle, tr, (7, 5, n), ns, ["diffCN_z"])


@pytest.mark.parametrize("n", [3, 5, 63, 64, 65, 255, 256, 257, 383, 384, 385, 512])
@pytest.mark.parametrize("shape", [0, 1])
def test_contiguous(pkg, oracle, tr, n, shape):  # noqa: F811
    sweeps(pkg, oracle, tr, (n, 5, 3), 3, ["diffCN_x"], part_shape_x=shape)


@pytest.mark.parametrize("box", [(2, 9, 3, 60, 2, 7), (1, 11, 1, 3, 1, 9), (5, 11, 2, 61, 3, 5)])
def test_boxes_and_masks(pkg, oracle, tr, box):  # noqa: F811
    st = pkg.workloads.random_state(11, 61, 9, 9, seed=3, latlon=True)
    st.bounds = box
    st.is_aloft = np.array([0, 1, 1, 0, 0, 1, 0, 1, 0], dtype=np.int32)
    st.dt *= 20.0
    a, b = st.copy(), st.copy()
    O, T = oracle.Oracle(a), tr.Transport(b)
    T.tune(line_solver="partitioned", jacobi_sweeps=0)
    for name in ("diffCN_x", "diffCN_y", "diffCN_z"):
        getattr(O, name)()
        getattr(T, name)()
    T.sync_to_host()
    T.close()
    assert_same(a, b, tol=TOL)
