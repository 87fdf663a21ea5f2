"""Partitioned solves of stiff dominant lines (factors of 1e9 and more): no
oracle comparison fits, since dgtsv's own error is as large, but the mass of
every line is kept to rounding.  With kappa as weights the matrix conserves a
line's mass, so its error is the weighted sum of the rows' residuals: per row
the right-hand side's three products and sums and a backward-stable solve's
residual, together taken as 64 ulps of (1 + L + R) max |q|."""
import numpy as np
import pytest

from test_gpu_parity import tr  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(3, 8, 9), (40, 65, 17), (127, 130, 4), (260, 5, 90)])
@pytest.mark.parametrize("scale", [1.0, 1.0e6, 1.0e11])
@pytest.mark.parametrize("dirn", [0, 1, 2])
def test_line_masses(pkg, tr, shape, scale, dirn):  # noqa: F811
    st = pkg.workloads.random_state(*shape, 2, seed=sum(shape), latlon=True)
    k = getattr(st, ("kx", "ky", "kz")[dirn])
    k *= scale
    inner = (slice(2, -2),) * 3
    kap = np.moveaxis(st.kappa_pd, dirn, 0)
    sig = np.moveaxis(getattr(st, ("sigma_nx_pd", "sigma_ny_pd", "sigma_nz_pd")[dirn]), dirn, 0)
    K = np.moveaxis(k, dirn, 0)[:, 1:-1, 1:-1]
    n = shape[dirn]
    cut = lambda a, lo, m: a[2 + lo:2 + lo + m, 2:-2, 2:-2]  # noqa: E731  (cells lo+1 .. lo+m)
    face = 0.5 * (K[:-1] + K[1:]) * (cut(sig, 0, n + 1) / (0.5 * (cut(kap, -1, n + 1) + cut(kap, 0, n + 1))))
    L = st.dt * face[:-1] * cut(sig, 0, n) / cut(kap, 0, n)
    R = st.dt * face[1:] * cut(sig, 1, n) / cut(kap, 0, n)
    before = np.moveaxis(st.concen_pd[inner][..., 0], dirn, 0).copy()
    T = tr.Transport(st)
    T.tune(line_solver="partitioned", jacobi_sweeps=0)
    getattr(T, "diffCN_" + "xyz"[dirn])()
    T.sync_to_host()
    T.close()
    after = np.moveaxis(st.concen_pd[inner][..., 0], dirn, 0)
    assert np.isfinite(after).all()
    w = cut(kap, 0, n)[..., None]
    error = np.abs((w * after).sum(0) - (w * before).sum(0))
    bound = 64 * 2.0 ** -53 * (np.abs(w) * (1.0 + np.abs(L) + np.abs(R))[..., None]).sum(0) * np.abs(before).max()
    assert (error <= bound).all(), (error / bound).max()
