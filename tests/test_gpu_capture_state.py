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
