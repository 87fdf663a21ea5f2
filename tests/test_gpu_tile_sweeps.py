"""The y and z sweeps in register tiles (csrc/advect_tile.hip): bitwise the
oracle on lines around the tile's cells (5 out of place, 6 and 8 in place)
and its workgroup's (20), on line counts around the 64 lanes, on bin counts
around a bin group (8), in place and out of place, through boxes, masks and
every limiter.  The tolerance is zero: the arithmetic is the reference's,
expression by expression."""
import numpy as np
import pytest

from test_gpu_parity import assert_same, run_both, tr  # noqa: F401

pytestmark = pytest.mark.gpu


def state(pkg, nx, ny, nz, ns, seed, **kw):
    return pkg.workloads.random_state(nx, ny, nz, ns, seed=seed, **kw)


@pytest.mark.parametrize("nx,ny,nz,ns", [(63, 4, 5, 1), (64, 5, 6, 7), (65, 6, 4, 8), (5, 19, 21, 9), (7, 20, 20, 2),
                                         (6, 21, 19, 17), (129, 41, 3, 3), (9, 3, 49, 5), (4, 66, 65, 2)])
@pytest.mark.parametrize("case", ["cartesian", "lonlat", "topo", "periodic"])
def test_sweeps_by_size(pkg, oracle, tr, nx, ny, nz, ns, case):  # noqa: F811
    kw = {"cartesian": {}, "lonlat": {"latlon": True}, "topo": {"zscaling_id": 2},
          "periodic": {"latlon": True, "periodic": True}}[case]
    st = state(pkg, nx, ny, nz, ns, nx + ny + nz, **kw)
    # the routines (in place and through ts1) and whole steps of both parities
    a, b = run_both(pkg, oracle, tr, st, [("AdvectHorz", 1), ("AdvectVert",), ("AdvectHorz", 2), ("advect_z",),
                                          ("advect_y",)])
    assert_same(a, b)
    for diffusion in (False, True):
        a, b = run_both(pkg, oracle, tr, st, [("transport_step", 1, diffusion), ("step_glue",),
                                              ("transport_step", 2, diffusion)])
        assert_same(a, b)


@pytest.mark.parametrize("lim", ["none", "laxwen", "bw", "fromm", "minmod", "superbee", "mc"])
@pytest.mark.parametrize("topo", [False, True])
def test_limiters(pkg, oracle, tr, lim, topo):  # noqa: F811
    st = state(pkg, 21, 23, 22, 3, 11, limiter=pkg.state.LIMITER_NAMES[lim], zscaling_id=2 if topo else 0)
    st.is_aloft = np.array([1, 0, 1], dtype=np.int32)
    a, b = run_both(pkg, oracle, tr, st, [("AdvectHorz", 1), ("AdvectVert",), ("AdvectHorz", 2)])
    assert_same(a, b)


@pytest.mark.parametrize("box", [(3, 60, 2, 20, 1, 12), (1, 70, 5, 25, 3, 20), (2, 69, 1, 24, 1, 22),
                                 (30, 33, 6, 8, 2, 22)])
def test_boxes(pkg, oracle, tr, box):  # noqa: F811
    st = state(pkg, 70, 25, 22, 3, 7, latlon=True)
    st.bounds = box
    a, b = run_both(pkg, oracle, tr, st, [("advect_y",), ("advect_z",)])
    assert_same(a, b)


def test_non_finite_winds(pkg, oracle, tr):  # noqa: F811
    """Infinite and NaN winds and concentrations spread as in the oracle."""
    st = state(pkg, 10, 12, 11, 2, 3)
    st.vy_pd[5, 6, 5] = np.inf
    st.vz_pd[7, 4, 6] = np.nan
    st.concen_pd[4, 8, 7, 0, :] = np.inf
    st.concen_pd[8, 3, 4, 1, :] = 1e308
    a, b = run_both(pkg, oracle, tr, st, [("AdvectHorz", 1), ("AdvectVert",)])
    assert_same(a, b)
