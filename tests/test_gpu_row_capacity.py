"""GPU test of cell-list rows that outgrow the ELL in a rebuild inside a step kernel, against the
oracle bit for bit: a minimisation that ends in exactly that step, and what the queries, a following
run and the pair lists then read; an NVE run through that step on the chunked loop.

A jittered square lattice with a wide skin: its first rows hold 12 entries, so the ELL starts
with 16 slots, and the first list rebuild (no cell sort) finds rows of more."""
import numpy as np
import pytest

from _helpers import oracle, pkg, workloads

P = pkg()
W = workloads()
pytestmark = pytest.mark.gpu

STATE = (P.F_X, P.F_Y, P.F_VX, P.F_VY, P.F_FX, P.F_FY, P.F_PE)


def lattice(g, phi):
    n, rng = g * g, np.random.default_rng(3)
    st = W.disk_config(n, phi, seed=3)
    k, h = rng.permutation(n), st.side / g
    st.x = (k % g + 0.5) * h + rng.uniform(-0.02, 0.02, n)
    st.y = (k // g + 0.5) * h + rng.uniform(-0.02, 0.02, n)
    return st


def make(st, be):
    return W.make_disk_system(P.System, st, W.neighbor_spec(st.side, skin=0.95), backend=be)


def fire(s, steps, dt=1e-2):
    return s.minimize_fire(P.fire_params(dt=dt, avg_pe_target=0.0, avg_pe_diff_target=0.0,
                                         fmax_target=0.0, max_steps=steps))


def state(s):
    return [s.download(f) for f in STATE]


def assert_same(a, b):
    for u, v in zip(a, b):
        assert np.array_equal(u, v)


def outgrows_in(st, steps, run):
    """On the oracle: the row capacity becomes 32 in step `steps`, by a list rebuild alone."""
    seen = []
    for k in (steps - 1, steps):
        s = make(st, oracle())
        run(s, k)
        q = s.neighbor_stats()
        seen.append((q["max_alloc"], q["n_rebuilds"], q["n_cell_rebuilds"]))
        s.close()
    return seen == [(16, 1, 1), (32, 2, 1)]


@pytest.mark.parametrize("g,phi,dt,steps", (
    (70, 0.90, 1e-2, 66),
    (70, 1.00, 1e-2, 59),
    (30, 1.00, 0.6, 11),    # a small system on the chunked loop (a short minimisation)
))
@pytest.mark.parametrize("then", ("queries", "forces", "pairs", "fire", "short fire", "nve"))
def test_minimisation_that_ends_in_the_outgrowing_step(g, phi, dt, steps, then):
    print("[gpu-case] rows outgrow in the last step", g, phi, steps, then, flush=True)
    st = lattice(g, phi)
    assert outgrows_in(st, steps, lambda s, k: fire(s, k, dt))
    got = []
    for be in (None, oracle()):
        s = make(st, be)
        r = fire(s, steps, dt)
        out = state(s) + [np.array([r.steps, r.avg_pe, r.fmax_sq])]
        if then == "queries":
            s.compute_stress()
            out += [s.download(f) for f in (P.F_STRESS_XX, P.F_STRESS_XY, P.F_STRESS_YY)]
            out += [s.reduce(q) for q in (P.RED_PRESSURE, P.RED_CONTACTS, P.RED_PE)]
            out += [s.download(P.F_CONTACTS)]
        elif then == "forces":
            s.zero_forces()
            s.compute_forces()
        elif then == "pairs":
            out += list(s.neighbor_pairs())
        elif then == "fire":
            fire(s, 40, dt)
        elif then == "short fire":
            for _ in range(3):
                fire(s, 1, dt)
        else:
            vx, vy = W.gaussian_velocities(st.n, 1e-4, 7)
            s.upload(P.F_VX, vx)
            s.upload(P.F_VY, vy)
            s.nve_run(0.01, 40)
        q = s.neighbor_stats()
        got.append(out + state(s) + [q["n_rebuilds"], q["n_cell_rebuilds"], q["total_entries"],
                                     q["max_alloc"]])
        s.close()
    assert_same(*got)


@pytest.mark.parametrize("steps", (35, 36, 37, 38, 70))
def test_nve_through_the_outgrowing_step(steps):
    print("[gpu-case] rows outgrow in an NVE step", steps, flush=True)
    st = lattice(70, 1.0)
    vx, vy = W.gaussian_velocities(st.n, 0.1, 5)

    def run(s, k):
        s.upload(P.F_VX, vx)
        s.upload(P.F_VY, vy)
        s.zero_forces()
        s.compute_forces()
        s.nve_run(0.01, k)

    assert outgrows_in(st, 36, run)
    got = []
    for be in (None, oracle()):
        s = make(st, be)
        run(s, steps)
        q = s.neighbor_stats()
        got.append(state(s) + [q["n_rebuilds"], q["n_cell_rebuilds"], q["total_entries"],
                               q["max_alloc"]])
        s.close()
    assert_same(*got)
