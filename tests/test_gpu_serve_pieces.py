"""GPU test of progress calls of any number of steps: one by one, more than a launch of resident
systems takes, and as good as unbounded (the call returns once everything has finished), with
resident systems alone and beside a rigid one, against the oracle bit for bit."""
import numpy as np
import pytest

from _helpers import oracle, pkg, workloads
from test_gpu_batch_sizes import alone, check, fire

P = pkg()
W = workloads()
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("beside", (False, True))
@pytest.mark.parametrize("steps", (1, 5000, 1 << 40))
def test_progress_of_any_length(steps, beside):
    print("[gpu-case] progress", steps, beside, flush=True)
    refs = [alone(n, 0.86, 70) for n in (256, 2049)]
    sv = P.Server(max_systems=4, arena_slots=1 << 13, budget_bytes=1 << 30,
                  vertex_slots=(1 << 13) if beside else 0)
    ids = [sv.submit(r[0].x, r[0].y, r[0].rad, r[0].mass, r[0].side,
                     P.jam_params(fire=fire(70)), mode=P.REQ_MINIMIZE) for r in refs]
    if beside:
        st = W.bumpy_config(64, 0.7, seed=5)
        s = W.make_bumpy_system(P.System, st, backend=oracle(), method=P.NBR_VERLET,
                                e_c=W.bumpy_contact_scale(st))
        s.minimize_fire(fire(70))
        rid = sv.submit(st.x, st.y, st.rad, st.mass, st.side, P.jam_params(fire=fire(70)),
                        e_c=W.bumpy_contact_scale(st), angle=st.angle,
                        vertices_per_particle=st.nverts, vertex_radius=st.rv,
                        mode=P.REQ_MINIMIZE)
    calls = 1
    while any(sv.progress(steps)[1:]):
        calls += 1
    assert steps == 1 or calls == 1
    for r, i in zip(refs, ids):
        got = sv.result(i)
        check(r, got["result"], got["x"], got["y"])
    if beside:
        assert np.array_equal(sv.result(rid)["x"], s.download(P.F_X))
    sv.close()
