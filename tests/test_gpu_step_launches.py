"""Launches a step does without (csrc/ash3d_tr.hip): the glue's ghost zeroing
stays pending over a source column (whose ghost cell above the top layer
counts as zero), captured steps hold neither the velocity ghosts nor, where
every line is dominant, the dgtsv-order alternative; bitwise the oracle's and
the eager steps' state."""
import numpy as np
import pytest

from test_gpu_parity import assert_same, tr  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_diffusion", [False, True])
@pytest.mark.parametrize("columns", [[(3, 4)], [(3, 4), (3, 4)], [(3, 4), (9, 2)], [(3, 4), (9, 2), (3, 4)]])
@pytest.mark.parametrize("then", ["step", "sync", "sweep", "subgrid"])
def test_sources_after_glue(pkg, oracle, tr, use_diffusion, columns, then):  # noqa: F811
    st = pkg.workloads.random_state(11, 9, 7, 3, seed=12, latlon=True)
    a, b = st.copy(), st.copy()
    O, T = oracle.Oracle(a), tr.Transport(b)
    T.tune(line_solver="exact")
    rng = np.random.default_rng(5)
    for S in (O, T):
        S.transport_step(1, use_diffusion)
        S.step_glue()
    for i, j in columns:
        f = rng.random((st.nz + 1, st.ns))
        O.source_column_add(i, j, f)
        T.source_column_add(i, j, f)
    if then == "step":
        for S in (O, T):
            S.transport_step(2, use_diffusion)
    elif then == "sweep":
        for S in (O, T):
            S.advect_z()
    elif then == "subgrid":
        for S in (O, T):
            S.transport_step_subgrid(2, use_diffusion, 3, 4, 2)
    T.sync_to_host()
    assert_same(a, b, names=("concen_pd", "outflow_xy1_pd", "outflow_xy2_pd", "outflow_xz1_pd"))
    T.close()


def test_replays_when_lines_or_winds_change(pkg, tr):  # noqa: F811
    """Replays after a wind upload, after diffusivities that leave lines not
    dominant (the dgtsv-order solves then run), and back."""
    st = pkg.workloads.random_state(21, 17, 10, 4, seed=33, latlon=True)
    st.concen_pd[..., 1] = st.concen_pd[..., 0]
    a, b = st.copy(), st.copy()
    E, G = tr.Transport(a), tr.Transport(b)
    for T in (E, G):
        T.step_glue()
        T.transport_step(1, True)
    G.graph_capture(2, True)
    G.graph_capture(3, True)
    itime = 2
    for change in ("none", "winds", "negative", "winds", "back", "none"):
        for X, T in ((a, E), (b, G)):
            if change == "winds":
                X.vx_pd *= 0.9
                X.vy_pd[2:-2, 2:-2, 2:-2] *= -0.8
                T.sync_from_host(tr.SYNC_WINDS)
            elif change == "negative":
                X.kx[5, 6, 4] = -abs(X.kx[5, 6, 4]) * 4.0
                X.kz[7, 8, 3] = -abs(X.kz[7, 8, 3]) * 4.0
                T.sync_from_host(tr.SYNC_DIFFK)
            elif change == "back":
                X.kx[...] = np.abs(X.kx)
                X.kz[...] = np.abs(X.kz)
                T.sync_from_host(tr.SYNC_DIFFK)
        for _ in range(2):
            E.step_glue()
            E.transport_step(itime, True)
            G.graph_launch(itime)
            itime += 1
        for T in (E, G):
            T.sync_to_host()
        assert np.array_equal(a.concen_pd, b.concen_pd), change
        assert np.array_equal(a.outflow_xy1_pd, b.outflow_xy1_pd), change
    E.close()
    G.close()
