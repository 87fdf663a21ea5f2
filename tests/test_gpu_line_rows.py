"""Row factors and line counts in one pass, and the factorisation left to
the device (csrc/diffuse.hip, k_line_rows and k_line_lu's gate).

The dgtsv-order solves read every number the pass and the factorisation
write, so bitwise equality with the oracle's sweeps pins them: line lengths
around a run of rows (8 and 16 runs per line, from 128 cells on) and line
counts around 64, after a partitioned sweep with the same time step left the
factorisation to the device, for matrices that do not need it, for nearly
singular ones that count as dominant, and for ones that are not dominant.
The partitioned sweeps themselves: 1e-12 of the largest value, the bar of
the other tests of those solves."""
import numpy as np
import pytest

from test_gpu_parity import assert_same, tr  # noqa: F401

pytestmark = pytest.mark.gpu

TOL = 1e-12
SHAPES = [(3, 8, 9), (7, 9, 17), (15, 16, 4), (127, 3, 8), (128, 4, 9), (5, 129, 7), (145, 5, 13), (4, 16, 131)]


def diffuse(T, O, names):
    for name in names:
        getattr(T, name)()
        getattr(O, name)()


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kind", ["dominant", "stiff", "negative"])
def test_exact_after_partitioned(pkg, oracle, tr, shape, kind):  # noqa: F811
    """Partitioned sweeps, then the dgtsv-order ones on the same factors from
    the initial state, then both again with another time step."""
    nx, ny, nz = shape
    st = pkg.workloads.random_state(nx, ny, nz, 3, seed=sum(shape), latlon=True)
    for k in (st.kx, st.ky, st.kz):
        k *= {"dominant": 1.0, "stiff": 1e11, "negative": 1.0}[kind]
        if kind == "negative":
            k[tuple(n // 2 for n in k.shape)] *= -3.0
    names = ["diffCN_x", "diffCN_y", "diffCN_z"]
    b = st.copy()
    T = tr.Transport(b)
    for scale in (1.0, 3.0):
        b.dt = st.dt * scale
        for solver in ("partitioned", "exact", "partitioned"):
            a = st.copy()
            a.dt = b.dt
            b.concen_pd[...] = st.concen_pd
            T.sync_from_host(tr.SYNC_CONCEN)
            T.tune(line_solver=solver, jacobi_sweeps=0)
            O = oracle.Oracle(a)
            diffuse(T, O, names)
            T.sync_to_host()
            if solver == "exact" or kind == "negative":
                assert_same(a, b)
            elif kind == "dominant":
                assert_same(a, b, tol=TOL)
    T.close()


def test_exact_steps_with_changing_dt(pkg, oracle, tr):  # noqa: F811
    """A new factorisation in every step, each solver in turn."""
    st = pkg.workloads.random_state(66, 31, 20, 4, seed=5, latlon=True)
    a, b = st.copy(), st.copy()
    O, T = oracle.Oracle(a), tr.Transport(b)
    for n, solver in enumerate(["exact", "partitioned", "exact", "partitioned", "partitioned"]):
        a.dt = b.dt = st.dt * (1.0 + 0.1 * n)
        T.tune(line_solver=solver)
        diffuse(T, O, ["diffCN_x", "diffCN_y", "diffCN_z"])
    T.sync_to_host()
    assert_same(a, b, tol=TOL)
    T.close()
