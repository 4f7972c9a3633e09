"""GPU tests of the batched engine at the sizes where its path changes, against the oracle bit for
bit: the resident classes' limits (256, 512, 1,024, 2,048 and 4,096 particles) and one particle
past each, the rule by which large or dense systems are resident beside many others or rigid ones
only, the per-phase kernels above 4,096 (with every workgroup size of the force pass), the
all-pairs row build above 16,384, and the same systems served."""
import numpy as np
import pytest

from _helpers import oracle, pkg, workloads

P = pkg()
W = workloads()
pytestmark = pytest.mark.gpu

EDGES = [n + k for n in (256, 512, 1024, 2048, 4096) for k in (0, 1)]


def fire(steps):
    return P.fire_params(avg_pe_target=0.0, avg_pe_diff_target=0.0, fmax_target=0.0,
                         max_steps=steps)


def threshold(cutoff):
    return 3.0 * 0.15 * 0.15 if cutoff == 1.7 else 3.0 * (0.5 * (cutoff - 1.4)) ** 2


_alone = {}


def alone(n, phi, steps, cutoff=1.7):
    """The system minimised alone by the oracle (Verlet method)."""
    key = (n, phi, steps, cutoff)
    if key not in _alone:
        st = W.disk_config(n, phi, seed=n)
        s = W.make_disk_system(P.System, st, W.NeighborSpec(P.NBR_VERLET, cutoff,
                                                            threshold(cutoff), 3, 1e30),
                               backend=oracle())
        r = s.minimize_fire(fire(steps))
        _alone[key] = (st, r.steps, s.reduce(P.RED_PE), s.reduce(P.RED_PRESSURE),
                       s.reduce(P.RED_CONTACTS), s.download(P.F_X), s.download(P.F_Y),
                       s.neighbor_stats()["n_rebuilds"])
        s.close()
    return _alone[key]


def check(ref, res, x, y):
    st, steps, pe, pressure, contacts, rx, ry, _ = ref
    assert (res.fire_steps_total, res.pe, res.pressure, res.contacts) == \
        (steps, pe, pressure, contacts), st.n
    assert np.array_equal(x, rx) and np.array_equal(y, ry), st.n


def minimise(refs, steps, block=None, graph=1, cutoff=1.7, rigid=None):
    b = P.Batch([r[0].n for r in refs] + ([rigid.n] if rigid else []),
                [0] * len(refs) + [rigid.nv] if rigid else None)
    b.config(1.0, 2.0, cutoff, threshold(cutoff))
    b.set_option(P.OPT_GRAPH, graph)
    if block:
        b.set_option(P.OPT_FORCE_BLOCK, block)
    for k, r in enumerate(refs):
        st = r[0]
        b.set_system(k, st.x, st.y, st.rad, st.mass, st.side)
    if rigid:
        b.set_rigid_system(len(refs), rigid.x, rigid.y, rigid.rad, rigid.mass, rigid.angle,
                           rigid.nverts, rigid.rv, rigid.side, e_c=W.bumpy_contact_scale(rigid))
    res, _ = b.minimize(fire(steps))
    for k, r in enumerate(refs):
        check(r, res[k], *b.get_system(k)[:2])
    b.close()


def test_resident_class_limits():
    refs = [alone(n, 0.86, 70) for n in EDGES]
    print("[gpu-case] batch minimise", EDGES, flush=True)
    assert min(r[-1] for r in refs) > 2
    minimise(refs, 70)
    for r in refs[::3]:
        minimise([r], 70)


def test_resident_class_limits_beside_a_rigid_system():
    """(Whose longer steps make the largest class resident.)"""
    refs = [alone(n, 0.86, 70) for n in EDGES]
    print("[gpu-case] batch minimise beside a rigid system", EDGES, flush=True)
    minimise(refs, 70, rigid=W.bumpy_config(64, 0.7, seed=5))


@pytest.mark.parametrize("cutoff", (1.7, 2.3))
@pytest.mark.parametrize("sizes", (
    (2049,), (4096,), (4000, 4096), (2049,) * 6, (64, 1000, 2000, 4096), (1000,), (2000,) * 3,
    (3000,) * 24,
))
def test_resident_rule(sizes, cutoff):
    print("[gpu-case] resident rule", sizes[:4], len(sizes), cutoff, flush=True)
    minimise([alone(n, 0.80, 50, cutoff) for n in sizes], 50, cutoff=cutoff)


@pytest.mark.parametrize("n", (257, 513, 1025, 2049, 4097))
def test_jams_past_a_limit(n):
    print("[gpu-case] batch jam", n, flush=True)
    st = W.disk_config(n, 0.80, seed=n)
    prm = P.jam_params(pressure_target=1e-2, window_rel=0.5, strain_step=2e-2,
                       max_compression_steps=12, fire=fire(40))
    s = W.make_disk_system(P.System, st, W.neighbor_spec(st.side, method=P.NBR_VERLET),
                           backend=oracle())
    r = s.jam(prm)
    b = P.Batch([n])
    b.set_system(0, st.x, st.y, st.rad, st.mass, st.side)
    res, _ = b.jam(prm)
    x, y, side = b.get_system(0)
    for f in ("status", "compression_steps", "fire_steps_total", "pressure", "packing_fraction",
              "pe", "box_length", "contacts"):
        assert getattr(res[0], f) == getattr(r, f), f
    assert np.array_equal(x, s.download(P.F_X)) and np.array_equal(y, s.download(P.F_Y))
    b.close()
    s.close()


@pytest.mark.parametrize("block", (64, 128, 256))
def test_force_pass_workgroups(block):
    """The workgroup sizes of the force pass, which disk systems above 4,096 particles take."""
    refs = [alone(n, 0.86, 70) for n in (4097, 4160, 300)] + [alone(6007, 0.86, 70)]
    print("[gpu-case] force pass workgroups", block, flush=True)
    minimise(refs, 70, block=block)


@pytest.mark.parametrize("graph", (0, 1))
def test_all_pairs_rows_above_16384(graph):
    refs = [alone(n, 0.86, 40) for n in (300, 16385, 4097, 16384)]
    print("[gpu-case] all-pairs rows", graph, flush=True)
    assert min(r[-1] for r in refs[1:]) > 1
    minimise(refs, 40, graph=graph)


def test_served_systems_past_the_limits():
    """A system above 16,384 particles comes and goes beside resident and per-phase ones."""
    order = [alone(n, 0.86, 40) for n in (300, 4097, 16385, 300, 16384, 4096)]
    print("[gpu-case] served", [r[0].n for r in order], flush=True)
    sv = P.Server(max_systems=4, arena_slots=1 << 15, budget_bytes=1 << 30, vertex_slots=0)
    ids = [sv.submit(r[0].x, r[0].y, r[0].rad, r[0].mass, r[0].side, P.jam_params(fire=fire(40)),
                     mode=P.REQ_MINIMIZE) for r in order]
    while any(sv.progress(16)[1:]):
        pass
    for r, i in zip(order, ids):
        got = sv.result(i)
        check(r, got["result"], got["x"], got["y"])



CROWD = (1, 2, 9, 64, 127, 128, 129, 300)


@pytest.mark.parametrize("count", (256, 257, 520))
def test_crowds_of_small_systems(count):
    """More small systems than CUs take the smallest class (and its neighbours the next)."""
    kinds = [alone(n, 0.84, 60) for n in CROWD]
    small = [r for r in kinds if r[0].n <= 128]
    print("[gpu-case] crowd", count, flush=True)
    minimise([small[k % len(small)] for k in range(count)] + kinds[-2:], 60)


def test_crowd_jams_and_is_served():
    prm = P.jam_params(pressure_target=1e-2, window_rel=0.5, strain_step=2e-2,
                       max_compression_steps=8, fire=fire(40))
    sts = [W.disk_config(n, 0.80, seed=n) for n in (20, 64, 100, 128)]
    ref = []
    for st in sts:
        s = W.make_disk_system(P.System, st, W.neighbor_spec(st.side, method=P.NBR_VERLET),
                               backend=oracle())
        ref.append((s.jam(prm), s.download(P.F_X)))
        s.close()
    print("[gpu-case] crowd jams", flush=True)
    b = P.Batch([sts[k % 4].n for k in range(300)])
    sv = P.Server(max_systems=300, arena_slots=1 << 16, budget_bytes=1 << 30, vertex_slots=0)
    ids = []
    for k in range(300):
        st = sts[k % 4]
        b.set_system(k, st.x, st.y, st.rad, st.mass, st.side)
        ids.append(sv.submit(st.x, st.y, st.rad, st.mass, st.side, prm))
    res, _ = b.jam(prm)
    while any(sv.progress(32)[1:]):  # (the crowd thins out: its systems change class)
        pass
    for k in range(300):
        got = sv.result(ids[k])
        for f in ("status", "compression_steps", "fire_steps_total", "pressure", "pe",
                  "contacts"):
            assert getattr(res[k], f) == getattr(ref[k % 4][0], f), (k, f)
            assert getattr(got["result"], f) == getattr(ref[k % 4][0], f), (k, f)
        assert np.array_equal(b.get_system(k)[0], ref[k % 4][1])
        assert np.array_equal(got["x"], ref[k % 4][1])
    b.close()
    sv.close()


@pytest.mark.parametrize("count", (512, 513))
def test_crowds_of_small_rigid_systems(count):
    """More small rigid systems than the row build has workgroups get all-pairs rows."""
    sts = [W.bumpy_config(n, 0.75, seed=n) for n in (2, 9, 30, 127, 128, 200)]
    ref = []
    for st in sts:
        s = W.make_bumpy_system(P.System, st, backend=oracle(), e_c=W.bumpy_contact_scale(st),
                                method=P.NBR_VERLET)
        r = s.minimize_fire(fire(40))
        ref.append((r.steps, s.reduce(P.RED_PE), s.download(P.F_X), s.download(P.F_ANGLE)))
        s.close()
    pick = [k % 4 for k in range(count)] + [4, 5]
    print("[gpu-case] rigid crowd", count, flush=True)
    b = P.Batch([sts[k].n for k in pick], [sts[k].nv for k in pick])
    for i, k in enumerate(pick):
        t = sts[k]
        b.set_rigid_system(i, t.x, t.y, t.rad, t.mass, t.angle, t.nverts, t.rv, t.side,
                           e_c=W.bumpy_contact_scale(t))
    res, _ = b.minimize(fire(40))
    for i, k in enumerate(pick):
        x, y, a = b.get_rigid_system(i)[:3]
        assert (res[i].fire_steps_total, res[i].pe) == ref[k][:2], sts[k].n
        assert np.array_equal(x, ref[k][2]) and np.array_equal(a, ref[k][3]), sts[k].n
    b.close()
