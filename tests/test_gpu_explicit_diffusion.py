"""Explicit diffusion sweeps (csrc/diffuse_explicit.hip) against the oracle,
bitwise: line lengths around the cells of a wave (8) and of a workgroup (64)
in y and z, x rows around one, two, four and eight cells per thread and
beyond a workgroup (8192), line counts around 64, bin counts around a group
(8), boxes, masks and periodic x; captured steps with explicit diffusion."""
import numpy as np
import pytest

from test_gpu_parity import assert_same, run_both, tr  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz,ns", [(63, 7, 9, 1), (64, 8, 8, 8), (65, 9, 7, 9), (3, 63, 65, 2), (5, 64, 64, 17),
                                         (2, 65, 129, 1), (257, 1, 3, 3), (513, 2, 1, 2), (1025, 3, 2, 1)])
@pytest.mark.parametrize("periodic", [False, True])
def test_sweeps_by_size(pkg, oracle, tr, nx, ny, nz, ns, periodic):  # noqa: F811
    st = pkg.workloads.random_state(nx, ny, nz, ns, seed=nx + ny, latlon=periodic, periodic=periodic, use_cn=False)
    a, b = run_both(pkg, oracle, tr, st, [("diff_x",), ("diff_y",), ("diff_z",)])
    assert_same(a, b)
    a, b = run_both(pkg, oracle, tr, st, [("transport_step", 1, True), ("step_glue",), ("transport_step", 2, True)])
    assert_same(a, b)


def test_rows_beyond_a_workgroup(pkg, oracle, tr):  # noqa: F811
    st = pkg.workloads.random_state(8200, 2, 2, 1, seed=3, latlon=True, periodic=True, use_cn=False)
    st.dt = 1e-6
    a, b = run_both(pkg, oracle, tr, st, [("diff_x",)])
    assert_same(a, b)


@pytest.mark.parametrize("box", [(3, 60, 2, 66, 1, 12), (1, 70, 5, 70, 3, 20), (30, 30, 64, 65, 2, 22)])
def test_boxes_and_masks(pkg, oracle, tr, box):  # noqa: F811
    st = pkg.workloads.random_state(70, 70, 22, 3, seed=7, latlon=True, use_cn=False)
    st.bounds = box
    st.is_aloft = np.array([1, 0, 1], dtype=np.int32)
    a, b = run_both(pkg, oracle, tr, st, [("diff_x",), ("diff_y",), ("diff_z",)])
    assert_same(a, b)


def test_captured_steps(pkg, oracle, tr):  # noqa: F811
    """Graphs captured with explicit diffusion replay to the eager bits."""
    st = pkg.workloads.random_state(33, 70, 12, 2, seed=9, latlon=True, use_cn=False)
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
