"""The kernels that read the whole state between steps -- output products,
column loads, mass totals, slab maxima, the met interpolation and the time
step -- against the oracle (bitwise) or, for the mass totals, numpy (1e-13
of each bin's sum of magnitudes: 1e5 rounded terms of about 1e-16 each), on
sizes around their tiles: 64 columns, 16 levels, groups of 8 bins, 64 rows,
384 columns."""
import numpy as np
import pytest

from test_gpu_driver import met_steps, params
from test_gpu_products import KEYS
from test_gpu_parity import tr  # noqa: F401

pytestmark = pytest.mark.gpu

SIZES = [(63, 1, 15, 1), (64, 2, 16, 7), (65, 3, 17, 8), (8, 65, 33, 9), (385, 4, 3, 2), (5, 128, 1, 17)]


@pytest.mark.parametrize("nx,ny,nz,ns", SIZES)
def test_reductions_by_size(pkg, oracle, tr, nx, ny, nz, ns):  # noqa: F811
    st = pkg.workloads.random_state(nx, ny, nz, ns, seed=nx + nz, latlon=True, diffusivity=False)
    st.concen_pd[..., 1] = st.concen_pd[..., 0]
    rng = np.random.default_rng(nz)
    st.deposit_granularity[...] = 10.0 * rng.random(st.deposit_granularity.shape)
    for name in ("outflow_yz1_pd", "outflow_yz2_pd", "outflow_xz1_pd", "outflow_xz2_pd", "outflow_xy2_pd"):
        getattr(st, name)[...] = rng.random(getattr(st, name).shape)
    dz = 0.3 + 0.1 * rng.random(nz)
    zcc = np.cumsum(dz) - 0.5 * dz
    b = st.copy()
    O, T = oracle.Oracle(st), tr.Transport(b)
    # products and column load
    kw = dict(cloudcon_thresh=20.0, cloudload_thresh=float(0.01 * nz), depo_thresh=float(2e-3 * ns))
    got, ref = T.products(dz, zcc, **kw), O.products(dz, zcc, **kw)
    for k in KEYS:
        assert np.array_equal(got[k], ref[k]), k
    assert got["cloud_area"] == ref["cloud_area"] and got["deposit_area"] == ref["deposit_area"]
    load = np.zeros((nx, ny))
    q = st.interior(1)
    for k in range(nz):
        s = np.zeros((nx, ny))
        for n in range(ns):
            s = s + q[:, :, k, n]
        load = load + s * dz[k] / 1.0e3
    assert np.array_equal(T.column_load(dz), load)
    # mass totals
    kap = st.kappa_pd
    I = np.s_[2:-2, 2:-2]
    aloft = np.einsum("ijkn,ijk->n", st.interior(), kap[2:-2, 2:-2, 2:-2])
    dep = np.einsum("ijn,ij->n", st.deposit_granularity, kap[2:-2, 2:-2, 1])
    out = sum(np.einsum("abn,ab->n", getattr(st, f"outflow_{nm}_pd")[I], kp) for nm, kp in
              (("yz1", kap[1][I]), ("yz2", kap[nx + 2][I]), ("xz1", kap[:, 1][I]), ("xz2", kap[:, ny + 2][I]),
               ("xy2", kap[:, :, nz + 2][I])))
    for g, r in zip(T.mass_totals(), (aloft, dep, out)):
        assert np.all(np.abs(g - r) <= 1e-13 * np.abs(r)), (g, r)
    # slab maxima: a small cloud away from the walls
    for h in (st, b):
        h.concen_pd[...] = 0.0
        h.concen_pd[2 + nx // 2, 2 + ny // 2, 2 + nz // 2, ns - 1, :] = 3.0
    T.sync_from_host(tr.SYNC_CONCEN)
    v = (max(1, nx // 3), max(1, ny // 3), 1)
    assert T.minmax_index(*v) == O.minmax_index(*v)[1]
    # met interpolation, then the time step from the interpolated winds
    if ns > 1:
        m = met_steps(st, 5)
        T.met_push(*m[0])
        T.met_push(*m[1])
        O.met_interp(m[0], m[1], 0.3, True)
        T.met_interp(0.3, True)
        kw = dict(is_latlon=1, n_gs_aloft=ns)
        dto, diago = O.adjust_dt(params(oracle.DtParams, dz, **kw))
        dtg, diagg = T.adjust_dt(params(tr.DtParams, dz, **kw))
        assert dtg == dto and np.array_equal(diagg, diago)
        T.sync_to_host(tr.SYNC_WINDS | tr.SYNC_VF)
        for name in ("vx_pd", "vy_pd", "vz_pd", "vf_pd"):
            assert np.array_equal(getattr(st, name)[2:-2, 2:-2, 2:-2], getattr(b, name)[2:-2, 2:-2, 2:-2]), name
    T.close()
