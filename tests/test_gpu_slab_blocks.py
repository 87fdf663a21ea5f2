"""The slab maxima behind minmax_index (csrc/meteo.hip) in the last block of
384 columns, of 64 rows, in the last level and bin: a cloud there alone decides
the box.  The oracle's box."""
import pytest

from test_gpu_parity import tr  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cell", [(384, 64, 5), (385, 65, 6), (430, 129, 7), (500, 130, 7), (499, 1, 1), (770, 70, 7)])
@pytest.mark.parametrize("b", [0, 2])
def test_clouds_in_the_last_blocks(pkg, oracle, tr, cell, b):  # noqa: F811
    nx = 500 if cell[0] <= 500 else 775
    st = pkg.workloads.random_state(nx, 130, 7, 3, seed=1)
    st.concen_pd[...] = 0.0
    st.concen_pd[cell[0] + 1, cell[1] + 1, cell[2] + 1, b, :] = 2.0
    O, T = oracle.Oracle(st.copy()), tr.Transport(st)
    for vent in ((2, 2, 2), (nx - 1, 128, 6)):
        assert T.minmax_index(*vent) == O.minmax_index(*vent)[1], vent
    T.close()
