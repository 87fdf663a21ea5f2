"""Sources on a periodic grid while the glue's ghost zeroing is pending (csrc/
ash3d_tr.hip, source_column_add): columns at both ends of the rows, whose ghost
copies Set_BC(1) and (2) write, then a step, a sweep, a read or a subgrid step.
Bitwise the oracle."""
import numpy as np
import pytest

from test_gpu_parity import assert_same, tr  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_diffusion", [False, True])
@pytest.mark.parametrize("columns", [[(1, 4)], [(11, 2), (11, 2)], [(1, 4), (11, 4)]])
@pytest.mark.parametrize("then", ["step", "read", "sweep", "subgrid"])
def test_sources_after_glue(pkg, oracle, tr, use_diffusion, columns, then):  # noqa: F811
    st = pkg.workloads.random_state(11, 9, 7, 3, seed=12, latlon=True, periodic=True)
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
    for S in (O, T):
        if then == "step":
            S.transport_step(2, use_diffusion)
        elif then == "sweep":
            S.advect_x()
        elif then == "subgrid":
            S.transport_step_subgrid(2, use_diffusion, 3, 4, 2)
    T.sync_to_host()
    assert_same(a, b, names=("concen_pd", "outflow_xy1_pd", "outflow_xy2_pd", "outflow_xz1_pd", "outflow_yz1_pd"))
    T.close()
