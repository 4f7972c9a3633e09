"""GPU test of the loops that hold a small disk system in one workgroup, against the oracle bit
for bit: sizes at the edges of a wave and of the size classes, both list methods, run lengths
around a launch's, cell sorts inside a run (static ids, Adam's moments), rows that outgrow the
ELL in the middle of a run, boxes too small for a cell grid, and overlaps too dense for the pair
list."""
import numpy as np
import pytest

from _helpers import oracle, pkg, workloads

P = pkg()
W = workloads()
pytestmark = pytest.mark.gpu

FIELDS = (P.F_X, P.F_Y, P.F_VX, P.F_VY, P.F_FX, P.F_FY, P.F_PE)
CELL, VERLET = P.NBR_CELL, P.NBR_VERLET


def pair(n, phi, method, seed=1, skin=0.3, jitter=None):
    out = []
    st = W.disk_config(n, phi, seed=seed)
    if jitter is not None:  # a jittered square lattice: short rows
        g, rng = int(np.ceil(np.sqrt(n))), np.random.default_rng(seed)
        k, h = np.arange(n), st.side / g
        st.x = (k % g + 0.5) * h + rng.uniform(-jitter, jitter, n)
        st.y = (k // g + 0.5) * h + rng.uniform(-jitter, jitter, n)
    for be in (None, oracle()):
        out.append(W.make_disk_system(P.System, st, W.neighbor_spec(st.side, skin=skin,
                                                                    method=method), backend=be))
    return out


def heat(systems, temperature, seed=1):
    for s in systems:
        vx, vy = W.gaussian_velocities(s.n, temperature, seed)
        s.upload(P.F_VX, vx)
        s.upload(P.F_VY, vy)
        s.zero_forces()
        s.compute_forces()


def same(g, o, what):
    for f in FIELDS:
        assert np.array_equal(g.download(f), o.download(f)), (what, f)
    gs, os_ = g.neighbor_stats(), o.neighbor_stats()
    for k in ("max_alloc", "total_entries", "n_rebuilds", "n_cell_rebuilds"):
        assert gs[k] == os_[k], (what, k)
    pairs = [sorted(zip(*(a.tolist() for a in s.neighbor_pairs()))) for s in (g, o)]
    assert pairs[0] == pairs[1], what


def fire(s, steps, fmax=0.0):
    return s.minimize_fire(P.fire_params(avg_pe_target=0.0, avg_pe_diff_target=0.0,
                                         fmax_target=fmax, max_steps=steps))


@pytest.mark.parametrize("method", (CELL, VERLET))
@pytest.mark.parametrize("n", (30, 64, 65, 256, 257, 512, 513, 1023, 1024, 1025, 2048, 2049))
def test_fire_then_nve(n, method):
    print("[gpu-case] resident", n, method, flush=True)
    g, o = pair(n, 0.84, method, seed=n)
    rg, ro = fire(g, 300), fire(o, 300)
    assert (rg.steps, rg.stopped, rg.converged) == (ro.steps, ro.stopped, ro.converged)
    assert (rg.avg_pe, rg.fmax_sq, rg.dt, rg.alpha) == (ro.avg_pe, ro.fmax_sq, ro.dt, ro.alpha)
    same(g, o, "fire")
    heat((g, o), 1e-2, n)
    for steps in (15, 16, 257):
        for s in (g, o):
            s.nve_run(0.01, steps)
        same(g, o, steps)


def test_converges_inside_a_launch():
    g, o = pair(200, 0.70, CELL, seed=4)
    rg, ro = fire(g, 5000, 1e-6), fire(o, 5000, 1e-6)
    assert rg.converged == ro.converged == 1 and rg.steps == ro.steps
    same(g, o, "fire")


@pytest.mark.parametrize("method", (CELL, VERLET))
def test_cell_sorts_inside_a_run(method):
    g, o = pair(324, 0.5, method, seed=3, jitter=0.1)
    for s in (g, o):
        for k in range(3):
            s.adam_step(k + 1, 1e-3)
    heat((g, o), 1.0, 3)
    for s in (g, o):
        s.nve_run(0.01, 600)
    same(g, o, "nve")
    assert method == VERLET or o.neighbor_stats()["n_cell_rebuilds"] > 10
    for s in (g, o):  # the moments went with their particles
        for k in range(3, 6):
            s.adam_step(k + 1, 1e-3)
    for f in (P.F_X, P.F_Y):
        assert np.array_equal(g.download(f), o.download(f))


@pytest.mark.parametrize("method", (CELL, VERLET))
def test_rows_outgrow_the_ell(method):
    g, o = pair(300, 0.6, method, seed=3, skin=0.6)
    assert o.neighbor_stats()["max_alloc"] == 16
    rg, ro = fire(g, 200), fire(o, 200)
    assert rg.steps == ro.steps and rg.avg_pe == ro.avg_pe
    same(g, o, "fire")
    g, o = pair(324, 0.6, method, seed=3, skin=0.95, jitter=0.05)
    assert o.neighbor_stats()["max_alloc"] <= 16
    heat((g, o), 2.0, 3)
    for s in (g, o):
        s.nve_run(0.01, 400)
    same(g, o, "nve")
    assert o.neighbor_stats()["max_alloc"] == 32


@pytest.mark.parametrize("n,phi,method,skin", (
    (12, 0.8, VERLET, 0.3),   # under three cutoffs a side
    (40, 0.8, CELL, 0.6),     # three cells a side
    (600, 1.3, CELL, 0.3),    # more pairs than the pair list holds
    (600, 1.3, VERLET, 0.3),
    (200, 0.9, VERLET, 1.5),  # near rows longer than the row table
    (1500, 1.3, CELL, 0.3),
))
def test_small_boxes_and_dense_systems(n, phi, method, skin):
    g, o = pair(n, phi, method, seed=2, skin=skin)
    rg, ro = fire(g, 120), fire(o, 120)
    assert rg.steps == ro.steps and rg.avg_pe == ro.avg_pe
    same(g, o, "fire")
    heat((g, o), 1e-1, 2)
    for s in (g, o):
        s.nve_run(0.005, 90)
    same(g, o, "nve")
