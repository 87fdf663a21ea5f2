"""Replays whose line factors were renewed since the capture (csrc/
ash3d_tr.hip, graph_launch): captures that leave out the dgtsv-order
alternative where every line is dominant replay the step that holds it until
the new lines are known to be dominant.  Eager steps take the same solvers
(no Jacobi sweeps), so the states agree bitwise; a replay does not wait for
the device."""
import time

import numpy as np
import pytest

from test_gpu_parity import tr  # noqa: F401

pytestmark = pytest.mark.gpu


def negative(X, axis, on):
    k = getattr(X, "k" + axis)
    c = tuple(n // 2 for n in k.shape)
    k[c] = -4.0 * abs(k[c]) if on else abs(k[c])


@pytest.mark.parametrize("solver", ["partitioned", "exact"])
def test_replays_after_each_change(pkg, tr, solver):  # noqa: F811
    """Lines of one direction at a time leave dominance and come back, also
    between the two parities' replays, and an eager step of another dt comes
    in between."""
    st = pkg.workloads.random_state(21, 17, 10, 4, seed=34, latlon=True)
    st.concen_pd[..., 1] = st.concen_pd[..., 0]
    a, b = st.copy(), st.copy()
    E, G = tr.Transport(a), tr.Transport(b)
    for T in (E, G):
        T.tune(line_solver=solver, jacobi_sweeps=0)
        T.step_glue()
        T.transport_step(1, True)
    for p in (2, 3):
        G.graph_capture(p, True)
    itime = 2
    for axis, on, replays, other_dt in (
            (None, 0, 4, 0), ("x", 1, 1, 0), ("z", 1, 2, 0), ("x", 0, 1, 0), (None, 0, 2, 1), ("y", 1, 3, 1),
            ("z", 0, 1, 0), ("y", 0, 1, 0), (None, 0, 4, 0), (None, 0, 3, 1)):
        for X, T in ((a, E), (b, G)):
            if axis:
                negative(X, axis, on)
                T.sync_from_host(tr.SYNC_DIFFK)
            if other_dt:
                X.dt *= 0.75
                T.step_glue()
                T.transport_step(itime, True)
                X.dt /= 0.75
        itime += bool(other_dt)
        for _ in range(replays):
            E.step_glue()
            E.transport_step(itime, True)
            G.graph_launch(itime)
            itime += 1
            for T in (E, G):
                T.sync_to_host()
            assert np.array_equal(a.concen_pd, b.concen_pd), (axis, on, itime)
            assert np.array_equal(a.outflow_xy1_pd, b.outflow_xy1_pd), (axis, on, itime)
    E.close()
    G.close()


def test_replay_does_not_wait(pkg, tr):  # noqa: F811
    """Steps of another dt are queued, then a replay, whose factors have to be
    renewed: it returns while the queue is being worked on."""
    st = pkg.workloads.random_state(160, 120, 50, 8, seed=35, latlon=True)
    T = tr.Transport(st)
    T.tune(line_solver="partitioned")
    dt = st.dt
    T.step_glue()
    T.transport_step(1, True)
    for p in (2, 3):
        T.graph_capture(p, True)
    best = 1.0e9
    for _ in range(3):
        st.dt = 0.5 * dt
        for itime in range(2, 42):
            T.step_glue()
            T.transport_step(itime, True)
        t0 = time.perf_counter()
        T.graph_launch(2)
        t1 = time.perf_counter()
        T.synchronize()
        best = min(best, (t1 - t0) / (time.perf_counter() - t0))
    assert best < 0.5, best
    T.close()
