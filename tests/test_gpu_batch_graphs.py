"""GPU test of the batched engine's launch graph, which is dropped while a batch lives (a system above
16,384 particles comes or goes in the serving loop; autotuning) and must not be destroyed again
with it: the calls after it see no stale error.  And what the autotuners leave alone."""
import pytest

from _helpers import pkg, workloads

P = pkg()
W = workloads()
pytestmark = pytest.mark.gpu


def fire(steps):
    return P.fire_params(avg_pe_target=0.0, avg_pe_diff_target=0.0, fmax_target=0.0,
                         max_steps=steps)


def rigid_batch(st):
    b = P.Batch([st.n], [st.nv])
    b.set_rigid_system(0, st.x, st.y, st.rad, st.mass, st.angle, st.nverts, st.rv, st.side,
                       e_c=W.bumpy_contact_scale(st))
    return b


def other_batch_runs():
    st = W.bumpy_config(64, 0.75, seed=1)
    b = rigid_batch(st)
    res, _ = b.minimize(fire(40))
    assert res[0].fire_steps_total == 40
    b.close()
    s = W.make_disk_system(P.System, W.disk_config(300, 0.8), None)
    s.nve_run(0.01, 3)
    s.close()


def test_large_system_leaves_the_server():
    print("[gpu-case] graph dropped by the server", flush=True)
    for keep in (False, True):  # the last graph dropped, or captured again
        sv = P.Server(max_systems=4, arena_slots=1 << 15, budget_bytes=1 << 30, vertex_slots=0)
        for n in (16385,) + ((5000,) if keep else ()):
            st = W.disk_config(n, 0.80, seed=n)
            sv.submit(st.x, st.y, st.rad, st.mass, st.side, P.jam_params(fire=fire(40)),
                      mode=P.REQ_MINIMIZE)
            while any(sv.progress(32)[1:]):
                pass
        sv.close()
        other_batch_runs()


def test_autotuned_batch_is_closed():
    print("[gpu-case] graph dropped by the autotuner", flush=True)
    b = rigid_batch(W.bumpy_config(64, 0.75, seed=1))
    prm = P.jam_params(pressure_target=1e-2, window_rel=0.5, strain_step=1e-2, fire=fire(64))
    b.autotune_shape(prm, trial_steps=32)
    b.close()
    other_batch_runs()


@pytest.mark.parametrize("block", (64, 128, 256))
def test_autotuners_leave_what_has_no_effect(block):
    """Resident systems alone take neither a launch length nor the force pass."""
    print("[gpu-case] autotune of resident systems", block, flush=True)
    prm = P.jam_params(pressure_target=1e-2, window_rel=0.5, strain_step=1e-2, fire=fire(64))
    b = P.Batch([200, 300])
    for k, n in enumerate((200, 300)):
        st = W.disk_config(n, 0.8, seed=n)
        b.set_system(k, st.x, st.y, st.rad, st.mass, st.side)
    b.set_option(P.OPT_FORCE_BLOCK, block)
    assert b.autotune(prm, trial_steps=64, cutoffs=(1.6, 1.9), chunks=(48, 8, 32))[1] == 48
    blk, pct, ms = b.autotune_shape(prm, trial_steps=64)
    assert blk == block and pct in (100, 125, 150) and 0 < ms < 1e3
    b.close()
    b = P.Batch([5000])  # the per-phase kernels: every candidate is timed
    st = W.disk_config(5000, 0.8, seed=1)
    b.set_system(0, st.x, st.y, st.rad, st.mass, st.side)
    assert b.autotune(prm, trial_steps=64, cutoffs=(1.6, 1.9), chunks=(8, 32))[1] in (8, 32)
    assert b.autotune_shape(prm, trial_steps=64)[0] in (64, 128, 256)
    b.close()
