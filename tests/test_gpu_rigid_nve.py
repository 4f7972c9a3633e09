"""GPU test of the device-resident NVE loop of rigid bumpy systems against the oracle, bit for
bit: run lengths around a chunk's, rotation on and off, both list methods, a system hot enough
for list rebuilds inside a chunk and cell sorts that halt one, particles with more vertices than
the one-pass force phase holds, and forces accumulated after a run without zeroing."""
import numpy as np
import pytest

from _helpers import oracle, pkg, workloads

P = pkg()
W = workloads()
pytestmark = pytest.mark.gpu

FIELDS = (P.F_X, P.F_Y, P.F_VX, P.F_VY, P.F_FX, P.F_FY, P.F_PE, P.F_ANGLE, P.F_OMEGA, P.F_TORQUE)


def pair(n, verts, method, rotation, temperature, seed):
    out = []
    st = W.bumpy_config(n, 0.72, seed=seed, n_small=verts[0], n_large=verts[1])
    vx, vy = W.gaussian_velocities(n, temperature, seed)
    for be in (None, oracle()):
        s = W.make_bumpy_system(P.System, st, backend=be, e_c=W.bumpy_contact_scale(st),
                                method=method, rotation=rotation)
        s.minimize_fire(P.fire_params(max_steps=20))
        s.upload(P.F_VX, vx)
        s.upload(P.F_VY, vy)
        s.upload(P.F_OMEGA, vx[::-1].copy())
        s.zero_forces()
        s.compute_forces()
        out.append(s)
    return out


@pytest.mark.parametrize("n,verts,method,rotation,temperature,runs", (
    (130, (20, 28), 3, True, 1e-4, (1, 2, 33, 34, 65)),
    (130, (20, 28), 2, False, 1e-4, (40, 3)),
    (1100, (20, 28), 2, True, 1e-4, (40,)),
    (700, (20, 28), 3, True, 4.0, (150, 31)),
    (70, (20, 900), 3, True, 1e-3, (35,)),
))
def test_runs_equal_the_oracle(n, verts, method, rotation, temperature, runs):
    print("[gpu-case] rigid nve", n, verts, method, rotation, temperature, flush=True)
    g, o = pair(n, verts, method, rotation, temperature, n)
    for steps in runs:
        for s in (g, o):
            s.nve_run(0.01, steps)
        for f in FIELDS:
            assert np.array_equal(g.download(f), o.download(f)), (steps, f)
    gs, os_ = g.neighbor_stats(), o.neighbor_stats()
    assert gs["n_rebuilds"] == os_["n_rebuilds"]
    assert gs["n_cell_rebuilds"] == os_["n_cell_rebuilds"]
    if temperature > 1.0:
        assert gs["n_cell_rebuilds"] > 2
    for s in (g, o):  # += onto the last step's forces
        s.compute_forces()
    for f in (P.F_FX, P.F_TORQUE, P.F_PE):
        assert np.array_equal(g.download(f), o.download(f)), f
