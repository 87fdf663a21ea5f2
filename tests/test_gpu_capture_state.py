"""What a capture leaves alone, and what it asks for (csrc/ash3d_tr.hip,
graph_capture): the velocity ghosts keep what was uploaded until a step or
replay runs Set_BC(1)."""
import numpy as np
import pytest

from test_gpu_parity import tr  # noqa: F401

pytestmark = pytest.mark.gpu

WINDS = ("vx_pd", "vy_pd", "vz_pd", "vf_pd")


@pytest.mark.parametrize("use_diffusion", [False, True])
@pytest.mark.parametrize("periodic", [False, True])
def test_captures_leave_velocity_ghosts(pkg, tr, use_diffusion, periodic):  # noqa: F811
    st = pkg.workloads.random_state(14, 9, 7, 2, seed=2, latlon=True, periodic=periodic)
    st.concen_pd[..., 1] = st.concen_pd[..., 0]
    a, b = st.copy(), st.copy()
    E, G = tr.Transport(a), tr.Transport(b)
    for T in (E, G):
        T.step_glue()
        T.transport_step(1, use_diffusion)
    rng = np.random.default_rng(6)
    new = {n: 5.0 * rng.standard_normal(getattr(a, n).shape) for n in WINDS}
    for X, T in ((a, E), (b, G)):
        for n, v in new.items():
            getattr(X, n)[...] = v
        T.sync_from_host(tr.SYNC_WINDS | tr.SYNC_VF)
    for p in (2, 3):
        G.graph_capture(p, use_diffusion)
    G.sync_to_host(tr.SYNC_WINDS | tr.SYNC_VF)
    for n, v in new.items():
        assert np.array_equal(getattr(b, n), v), n
    for itime in (2, 3, 4):  # and the replays run it
        E.step_glue()
        E.transport_step(itime, use_diffusion)
        G.graph_launch(itime)
    E.sync_to_host()
    G.sync_to_host()
    for n in WINDS + ("concen_pd", "outflow_yz1_pd", "outflow_xz2_pd", "outflow_xy1_pd"):
        assert np.array_equal(getattr(a, n), getattr(b, n)), n
    E.close()
    G.close()


def test_captures_follow_an_eager_diffusion(pkg, tr):  # noqa: F811
    """Explicit diffusion: refused before an x sweep on the present geometry
    and diffusivities, as a theta-scheme step's capture is."""
    st = pkg.workloads.random_state(14, 9, 7, 2, seed=2, latlon=True, use_cn=False)
    st.dt *= 0.2
    with tr.Transport(st) as T:
        T.transport_step(1, False)
        with pytest.raises(tr.Ash3dError, match="capture after an eager step"):
            T.graph_capture(2, True)
        T.graph_capture(2, False)
        T.diff_x()
        T.graph_capture(2, True)
        T.sync_from_host(tr.SYNC_DIFFK)
        with pytest.raises(tr.Ash3dError, match="capture after an eager step"):
            T.graph_capture(2, True)
        T.step_glue()
        T.transport_step(3, True)
        T.graph_capture(2, True)
        T.graph_launch(2)
        T.synchronize()


@pytest.mark.parametrize("change", ["box", "dt"])
def test_captures_leave_later_sweeps_right(pkg, oracle, tr, change):  # noqa: F811
    """A capture whose line factors are not the cached ones (another box or
    time step came before) forms them at once: eager sweeps after it, and
    replays of either parity first, are bitwise the oracle's."""
    st = pkg.workloads.random_state(18, 7, 16, 2, seed=8, latlon=True)
    st.concen_pd[..., 1] = st.concen_pd[..., 0]
    a, b = st.copy(), st.copy()
    O, T = oracle.Oracle(a), tr.Transport(b)
    T.tune(line_solver="exact")
    for S, h in ((O, a), (T, b)):
        S.transport_step(1, True)
        if change == "box":
            h.bounds = (3, 9, 2, 5, 4, 11)
            for name in ("diffCN_x", "diffCN_y", "diffCN_z"):
                getattr(S, name)()
            h.bounds = (1, 18, 1, 7, 1, 16)
        else:
            h.dt *= 0.7
    T.graph_capture(2, True)
    T.graph_capture(3, True)
    for S in (O, T):
        S.DiffuseVert()
        S.DiffuseHorz(1)
    for itime in (3, 2):
        O.step_glue()
        O.transport_step(itime, True)
        T.graph_launch(itime)
    T.sync_to_host()
    for n in ("concen_pd", "outflow_yz1_pd", "outflow_xz2_pd", "outflow_xy1_pd"):
        assert np.array_equal(getattr(a, n), getattr(b, n)), n
    T.close()
