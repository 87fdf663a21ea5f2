"""y and z sweeps in place in register tiles (csrc/advect_tile.hip) at the
edges of their rule: five, six or eight cells per wave by line length, the
largest workgroups (12 waves of five cells, 8 of six or eight), lines that
the streamed kernel keeps (more than 64 cells, few bins on many lines, many
bins on long lines).  Bitwise the oracle; the rule's bounds in line counts are
met with small lines on both sides."""
import numpy as np
import pytest

from test_gpu_parity import assert_same, run_both, tr  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 5, 6, 20, 21, 24, 25, 32, 33, 40, 41, 47, 48, 49, 55, 59, 60, 61, 64, 65])
@pytest.mark.parametrize("ns", [1, 3, 13])
@pytest.mark.parametrize("topo", [False, True])
def test_line_lengths(pkg, oracle, tr, N, ns, topo):  # noqa: F811
    kw = dict(latlon=True, zscaling_id=2 if topo else 0)
    mask = np.array(([1, 0, 1] * ns)[:ns], dtype=np.int32)
    st = pkg.workloads.random_state(67, N, 3, ns, seed=N + ns, **kw)
    st.is_aloft = mask
    a, b = run_both(pkg, oracle, tr, st, [("advect_y",), ("advect_y",)])
    assert_same(a, b)
    st = pkg.workloads.random_state(67, 3, N, ns, seed=N + ns, **kw)
    st.is_aloft = mask
    a, b = run_both(pkg, oracle, tr, st, [("advect_z",), ("AdvectVert",)])
    assert_same(a, b)


@pytest.mark.parametrize("shape,ns", [((64, 767, 21), 1), ((64, 768, 21), 1), ((64, 768, 20), 1), ((64, 1023, 33), 2),
                                      ((64, 1024, 33), 2), ((64, 1024, 33), 4), ((64, 1024, 33), 3), ((64, 1024, 32), 2),
                                      ((64, 511, 33), 8), ((64, 512, 33), 8), ((64, 1024, 49), 13), ((64, 1023, 49), 13)])
def test_line_counts(pkg, oracle, tr, shape, ns):  # noqa: F811
    st = pkg.workloads.random_state(*shape, ns, seed=ns, latlon=True)
    a, b = run_both(pkg, oracle, tr, st, [("advect_z",)])
    assert_same(a, b)
