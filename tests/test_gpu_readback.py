"""Reading the state back (csrc/host_state.hip): levels below and above the
size from which host threads write the ts1 level, the three forms of that
level (ts0's interior after a sweep, zero after the glue, as uploaded), rows
of odd length, one processor only (everything is copied), pageable and pinned
arrays; bitwise the oracle's two levels."""
import os

import numpy as np
import pytest
import torch

from test_gpu_parity import assert_same, tr  # noqa: F401

pytestmark = pytest.mark.gpu

SHAPES = [(9, 8, 7, 2), (97, 61, 45, 7), (97, 61, 45, 8), (130, 45, 20, 25), (20000, 3, 2, 4)]


def pinned(a):
    h = torch.empty(a.size, dtype=torch.float64, pin_memory=True).numpy().reshape(a.shape, order="F")
    h[...] = a
    return h


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("how", ["pageable", "pinned", "one processor"])
def test_levels(pkg, oracle, tr, shape, how):  # noqa: F811
    st = pkg.workloads.random_state(*shape, seed=sum(shape), latlon=True)
    a, b = st.copy(), st.copy()
    if how == "pinned":
        b.concen_pd = pinned(b.concen_pd)
    O, T = oracle.Oracle(a), tr.Transport(b)
    cpus = os.sched_getaffinity(0)
    try:
        if how == "one processor":
            os.sched_setaffinity(0, {min(cpus)})
        T.sync_to_host()  # as uploaded
        assert_same(a, b)
        for _ in range(2):  # a second time into memory that was written before
            O.advect_z()
            T.advect_z()
            T.sync_to_host()
            assert_same(a, b)
        b.concen_pd[...] = -1.0
        T.step_glue()
        T.sync_to_host()
    finally:
        os.sched_setaffinity(0, cpus)
    assert np.array_equal(b.concen_pd[..., 1], np.zeros_like(b.concen_pd[..., 1]))
    assert np.array_equal(b.concen_pd[..., 0], a.concen_pd[..., 1])
    T.close()
