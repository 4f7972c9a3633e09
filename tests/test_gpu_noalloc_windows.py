"""GPU test of dpm_disk_forces_noalloc on particles with more pairs than a workgroup's LDS holds,
which are taken by windows of the index: indices in random order, in the order of the positions
(a particle's pairs are runs of indices) and in clusters, against the list-based entry points bit
for bit, in both grids."""
import numpy as np
import pytest

from _helpers import workloads
from test_gpu_noalloc_sizes import bare, listed

W = workloads()
pytestmark = pytest.mark.gpu


def config(n, phi, order, seed):
    st = W.disk_config(n, phi, seed=seed)
    rng = np.random.default_rng(seed)
    if order == "cluster":      # up to some 190 pairs, and particles with none
        st.side *= 4.0
        st.x = st.side / 2 + rng.normal(0.0, 0.02 * st.side, n)
        st.y = st.side / 2 + rng.normal(0.0, 0.02 * st.side, n)
    elif order == "sorted":
        k = np.lexsort((st.x, np.floor(st.y / 1.7)))
        st.x, st.y = st.x[k], st.y[k]
    elif order == "point":      # every particle a pair of every other
        st.side = 40.0
        st.x, st.y = 20.0 + rng.uniform(-0.4, 0.4, n), 20.0 + rng.uniform(-0.4, 0.4, n)
    return st


@pytest.mark.parametrize("n,phi,cutoff,order", (
    (33, 0.8, 1.7, "point"),        # 32 pairs each: as many as LDS holds
    (34, 0.8, 1.7, "point"),        # 33
    (300, 0.8, 1.7, "point"),
    (500, 0.85, 5.0, "random"),
    (2000, 0.85, 3.5, "random"),
    (2000, 0.85, 3.5, "sorted"),
    (3000, 0.85, 1.7, "cluster"),
    (8192, 3.0, 1.7, "sorted"),
    (8193, 0.85, 3.5, "random"),
    (8193, 0.85, 3.5, "sorted"),
    (9001, 0.85, 1.7, "cluster"),
    (50021, 0.85, 4.1, "sorted"),
))
def test_equals_the_list_path(n, phi, cutoff, order):
    print("[gpu-case] noalloc windows", n, phi, cutoff, order, flush=True)
    st = config(n, phi, order, n)
    got, ref = bare(st, cutoff, graph=n == 2000), listed(st, cutoff)
    for a, b, name in zip(got, ref, ("fx", "fy", "pe", "total")):
        assert np.array_equal(a, b), name
    assert np.max(np.abs(got[0])) > 0
