"""GPU test of the chunked FIRE loop of large disk systems against the oracle, bit for bit: sizes
around the decision kernel's workgroup sizes and stretch, list rebuilds inside a step (cell
lists) and rows that outgrow the ELL there."""
import numpy as np
import pytest

from _helpers import oracle, pkg, workloads

P = pkg()
W = workloads()
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,phi,skin,steps", (
    (4900, 0.90, 0.95, 300),    # a square lattice whose rows outgrow the ELL
    (4900, 1.00, 0.95, 300),
    (4096, 0.86, 0.3, 120),
    (32768, 0.84, 0.3, 60),     # 512 chunks
    (32769, 0.84, 0.3, 60),
    (131073, 0.84, 0.3, 60),    # more chunks than a stretch holds
))
def test_fire_equals_the_oracle(n, phi, skin, steps):
    print("[gpu-case] fire loop", n, phi, skin, steps, flush=True)
    st = W.disk_config(n, phi, seed=3)
    if skin > 0.3:
        g, rng = 70, np.random.default_rng(3)
        k, h = rng.permutation(n), st.side / g
        st.x = (k % g + 0.5) * h + rng.uniform(-0.02, 0.02, n)
        st.y = (k // g + 0.5) * h + rng.uniform(-0.02, 0.02, n)
    out = []
    for be in (None, oracle()):
        s = W.make_disk_system(P.System, st, W.neighbor_spec(st.side, skin=skin), backend=be)
        r = s.minimize_fire(P.fire_params(avg_pe_target=0.0, avg_pe_diff_target=0.0,
                                          fmax_target=0.0, max_steps=steps))
        assert skin == 0.3 or be is None or s.neighbor_stats()["max_alloc"] == 32
        out.append(([s.download(f) for f in (P.F_X, P.F_Y, P.F_FX, P.F_FY, P.F_PE)],
                    (r.steps, r.avg_pe, r.fmax_sq, r.dt, r.alpha), s.neighbor_stats()))
    (ga, gr, gs), (oa, orr, os_) = out
    assert gr == orr
    assert gs == os_ and os_["n_rebuilds"] > os_["n_cell_rebuilds"] > 0
    for a, b in zip(ga, oa):
        assert np.array_equal(a, b)
