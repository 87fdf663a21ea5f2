"""Adjust_DT's maxima (csrc/meteo.hip) where rows are packed into waves (a
fifth of the lanes or more idle by rows) and where they are not, and for every
size of the last group of bins; the largest wind, fall speed and smallest
diffusion time sit in the last cell or bin.  Bitwise the oracle's."""
import numpy as np
import pytest

from test_gpu_driver import met_steps, params
from test_gpu_parity import tr  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(3, 4, 5), (30, 7, 3), (51, 5, 4), (52, 5, 4), (63, 3, 5), (64, 3, 4), (65, 5, 3),
                                      (102, 3, 4), (103, 3, 4), (129, 2, 3)])
@pytest.mark.parametrize("ns", [1, 2, 3, 4, 5, 8, 9, 10, 12, 13])
def test_adjust_dt(pkg, oracle, tr, nx, ny, nz, ns):  # noqa: F811
    st = pkg.workloads.random_state(nx, ny, nz, ns, seed=nx + ns, latlon=True)
    st.vf_pd[1 + nx, 1 + ny, 1 + nz, ns - 1] = -900.0
    st.vx_pd[1 + nx, 1 + ny, 1 + nz] = 700.0
    st.kx[nx, ny, nz] *= 50.0
    m = met_steps(st, 5)
    O, T = oracle.Oracle(st), tr.Transport(st.copy())
    T.met_push(*m[0])
    T.met_push(*m[1])
    dz = np.linspace(0.4, 0.6, nz)
    for use_met in (0, 1):
        for latlon in (0, 1):
            kw = dict(is_latlon=latlon, n_gs_aloft=ns, use_met_next=use_met, use_diffusion=1)
            dto, diago = O.adjust_dt(params(oracle.DtParams, dz, **kw), m[1])
            dtg, diagg = T.adjust_dt(params(tr.DtParams, dz, **kw))
            assert dtg == dto and np.array_equal(diagg, diago)
    T.close()
