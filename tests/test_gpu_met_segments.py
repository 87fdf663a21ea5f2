"""Met interpolation by segments of an x row (csrc/meteo.hip): rows around 64
and 256 cells and their multiples, with and without the fall speeds.  Bitwise
the oracle's."""
import numpy as np
import pytest

from test_gpu_driver import met_steps
from test_gpu_parity import tr  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx", [2, 63, 64, 65, 127, 129, 255, 256, 257, 320, 512, 513, 700])
@pytest.mark.parametrize("use_vf", [False, True])
def test_met_interp(pkg, oracle, tr, nx, use_vf):  # noqa: F811
    st = pkg.workloads.random_state(nx, 5, 3, 2, seed=nx, latlon=True)
    a, b = st.copy(), st.copy()
    m = met_steps(st, 6)
    O, T = oracle.Oracle(a), tr.Transport(b)
    T.met_push(*m[0])
    T.met_push(*m[1])
    O.met_interp(m[0], m[1], 0.3, use_vf)
    T.met_interp(0.3, use_vf)
    T.sync_to_host(tr.SYNC_WINDS | tr.SYNC_VF)
    for name in ("vx_pd", "vy_pd", "vz_pd", "vf_pd"):
        assert np.array_equal(getattr(a, name), getattr(b, name)), name
    T.close()
