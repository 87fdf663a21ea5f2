"""dgtsv-order line solves without row interchanges (csrc/cn_exact.hip) and
the choice between them and the general kernels, bitwise the oracle: line
lengths around a chunk (8 rows), line counts around 64, one to nine bins
(one, two and four waves per workgroup), boxes, masks, periodic x; sweeps
whose elimination interchanges rows of matrices that are dominant row by
row; several sweeps, so that the choice is made on the device (the first
after a factorisation) and on the host (later ones), and captured."""
import numpy as np
import pytest

from test_gpu_parity import assert_same, run_both, tr  # noqa: F401

pytestmark = pytest.mark.gpu

SWEEPS = [("diffCN_x",), ("diffCN_y",), ("diffCN_z",)]


@pytest.mark.parametrize("nx,ny,nz,ns", [(7, 8, 9, 1), (63, 15, 2, 2), (64, 16, 17, 3), (65, 3, 8, 4), (2, 33, 32, 5),
                                         (31, 130, 7, 9), (129, 5, 25, 8)])
@pytest.mark.parametrize("periodic", [False, True])
def test_sweeps_by_size(pkg, oracle, tr, nx, ny, nz, ns, periodic):  # noqa: F811
    st = pkg.workloads.random_state(nx, ny, nz, ns, seed=nx + ny, latlon=periodic, periodic=periodic)
    a, b = run_both(pkg, oracle, tr, st, SWEEPS + SWEEPS + SWEEPS)
    assert_same(a, b)


@pytest.mark.parametrize("box", [(3, 60, 2, 30, 1, 12), (1, 70, 5, 31, 3, 20), (30, 32, 8, 10, 2, 22)])
@pytest.mark.parametrize("theta", [0.0, 0.5, 1.0])
def test_boxes_masks_theta(pkg, oracle, tr, box, theta):  # noqa: F811
    st = pkg.workloads.random_state(70, 33, 22, 5, seed=7, latlon=True, imp_fac=theta)
    st.bounds = box
    st.is_aloft = np.array([1, 0, 1, 1, 0], dtype=np.int32)
    a, b = run_both(pkg, oracle, tr, st, SWEEPS + SWEEPS)
    assert_same(a, b)


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_dominant_rows_with_interchanges(pkg, oracle, tr, axis):  # noqa: F811
    """Volumes that drop along a line make the next row's sub-diagonal entry
    larger than the pivot, although every row is dominant."""
    st = pkg.workloads.random_state(12, 11, 13, 3, seed=4)
    shape = [1, 1, 1]
    shape[axis] = st.kappa_pd.shape[axis]
    st.kappa_pd *= np.where(np.arange(shape[axis]) % 5 == 3, 1e-3, 1.0).reshape(shape)
    for k in (st.kx, st.ky, st.kz):
        k *= 50.0
    a, b = run_both(pkg, oracle, tr, st, SWEEPS + SWEEPS + SWEEPS)
    assert_same(a, b)


def test_captured_steps(pkg, oracle, tr):  # noqa: F811
    st = pkg.workloads.random_state(33, 20, 12, 4, seed=9, latlon=True)
    E, G = tr.Transport(st.copy()), tr.Transport(st.copy())
    for T in (E, G):
        T.transport_step(1, True)
    for it in (2, 3):
        G.graph_capture(it, True)
    for it in range(2, 8):
        E.step_glue()
        E.transport_step(it, True)
        G.graph_launch(it)
    for T in (E, G):
        T.sync_to_host()
    assert_same(E.st, G.st)
    E.close()
    G.close()


@pytest.mark.parametrize("n", [2, 8, 9, 56, 57, 63, 64, 65, 72, 73, 79, 80, 81])
@pytest.mark.parametrize("ns", [1, 2, 5])
def test_kept_right_hand_sides(pkg, oracle, tr, n, ns):  # noqa: F811
    """Lines whose eliminated right-hand sides stay in registers (up to 64
    and up to 80 cells) and longer ones; a box inside longer lines."""
    for shape, box in (((9, n, 4), None), ((7, 5, n), None), ((5, 90, 85), (1, 5, 4, 3 + n, 2, 1 + n))):
        st = pkg.workloads.random_state(*shape, ns, seed=n + ns, latlon=True)
        if box:
            st.bounds = box
        st.dt *= 30.0
        a, b = run_both(pkg, oracle, tr, st, [("diffCN_y",), ("diffCN_z",)] * 3)
        assert_same(a, b)
