"""Products and column loads of few bins on many columns (csrc/products.hip):
a thread per column, eight levels at a time, on both sides of the rule (four
bins, 2^17 columns), for levels around a group of eight.  Bitwise the oracle's
products, the loads bitwise the products'."""
import numpy as np
import pytest

from test_gpu_parity import tr  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(512, 256), (513, 257), (331, 397), (331, 395)])
@pytest.mark.parametrize("nz,ns", [(1, 1), (7, 2), (8, 4), (9, 3), (17, 1), (8, 5)])
def test_products(pkg, oracle, tr, nx, ny, nz, ns):  # noqa: F811
    st = pkg.workloads.random_state(nx, ny, nz, ns, seed=nz + ns, latlon=True)
    st.concen_pd[..., 1] = st.concen_pd[..., 0]
    rng = np.random.default_rng(3)
    st.deposit_granularity[...] = rng.random(st.deposit_granularity.shape)
    dz = np.linspace(0.4, 0.6, nz)
    zcc = np.cumsum(dz) - 0.5 * dz
    # thresholds inside the values, so that every branch is taken
    kw = dict(cloudcon_thresh=float(np.median(st.concen_pd[2:-2, 2:-2, 2:-2].sum(axis=3))), cloudload_thresh=1.0e-3)
    O, T = oracle.Oracle(st), tr.Transport(st.copy())
    want, got = O.products(dz, zcc, **kw), T.products(dz, zcc, **kw)
    for name in want:
        assert np.array_equal(np.asarray(want[name]), np.asarray(got[name])), name
    T.advect_z()
    load = T.column_load(dz)
    assert np.array_equal(load, T.products(dz, zcc, cloudload_thresh=-1.0e300)["cloud_load"])
    T.close()
