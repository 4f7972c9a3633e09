"""GPU test of rebuild thresholds at the ends of their range in the one-workgroup loops, against the
oracle bit for bit: never (an infinite or undefined threshold), at every step (zero or negative)
and rarely."""
import numpy as np
import pytest

from _helpers import oracle, pkg, workloads
from test_gpu_resident import fire, heat, same

P = pkg()
W = workloads()
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("thr", (float("nan"), float("inf"), 0.0, -1.0, 1e-300, 1.0))
@pytest.mark.parametrize("n,method", ((100, P.NBR_VERLET), (300, P.NBR_VERLET),
                                      (100, P.NBR_CELL), (300, P.NBR_CELL)))
def test_thresholds(n, method, thr):
    print("[gpu-case] threshold", n, method, thr, flush=True)
    st = W.disk_config(n, 0.6, seed=n)
    spec = W.neighbor_spec(st.side, method=method)
    spec.disp_thresh_sq, spec.cell_disp_thresh_sq = thr, 1e30
    g, o = (W.make_disk_system(P.System, st, spec, backend=be) for be in (None, oracle()))
    rg, ro = fire(g, 100), fire(o, 100)
    assert (rg.steps, rg.avg_pe) == (ro.steps, ro.avg_pe)
    heat((g, o), 1.0, n)
    for s in (g, o):
        s.nve_run(0.01, 60)
    same(g, o, thr)
    assert np.max(np.abs(o.download(P.F_X) - st.x)) > 0.3
