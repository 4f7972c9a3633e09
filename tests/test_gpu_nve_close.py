"""GPU test of the closing force of an NVE run on the chunked loop (every workgroup applies it,
whenever it starts) against the oracle, bit for bit: thousands of short runs, whose errors stay in
the velocities, at sizes of a few to some thousand workgroups."""
import numpy as np
import pytest

from _helpers import oracle, pkg, workloads

P = pkg()
W = workloads()
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,runs,steps", ((1600, 3000, 1), (4900, 3000, 1), (4900, 1000, 3),
                                          (20000, 600, 2), (600000, 6, 2)))
def test_short_runs_close_everywhere(n, runs, steps):
    print("[gpu-case] nve closes", n, runs, steps, flush=True)
    st = W.disk_config(n, 0.80, seed=n)
    vx, vy = W.gaussian_velocities(n, 1e-4, n)
    out = []
    for be in (None, oracle()):
        s = W.make_disk_system(P.System, st, W.neighbor_spec(st.side), backend=be)
        s.upload(P.F_VX, vx)
        s.upload(P.F_VY, vy)
        s.zero_forces()
        s.compute_forces()
        for _ in range(runs):
            s.nve_run(0.001, steps)
        out.append([s.download(f) for f in (P.F_X, P.F_Y, P.F_VX, P.F_VY, P.F_FX, P.F_FY,
                                            P.F_PE)])
        s.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b), int(np.sum(a != b))
