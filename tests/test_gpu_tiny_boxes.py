"""GPU test of rigid bumpy systems in boxes under a few particle diameters a side, where another
image of a ring can be nearer to a vertex than the nearest image of the ring's centre: vertex rows
entry by entry in row order and one evaluation against the oracle, and minimisations of the
batched engine and the serving loop against the oracle's, bit for bit."""
import numpy as np
import pytest

from _helpers import oracle, pkg, workloads

P = pkg()
W = workloads()
pytestmark = pytest.mark.gpu

SYSTEMS = [(n, phi) for n in (1, 2, 3, 4, 5, 7, 9, 12) for phi in (0.6, 0.84, 1.0, 1.3)]


def rows(s):
    i, j = s.vertex_pairs()
    o = np.argsort(i, kind="stable")
    return [i[o], j[o]]


def spec():
    return P.fire_params(avg_pe_target=0.0, avg_pe_diff_target=0.0, fmax_target=0.0,
                         max_steps=40)


@pytest.mark.parametrize("n,phi", SYSTEMS)
@pytest.mark.parametrize("n_small,n_large", ((20, 28), (9, 14), (33, 40)))
def test_rows_and_forces(n, phi, n_small, n_large):
    print("[gpu-case] tiny box rows", n, phi, n_small, n_large, flush=True)
    for seed in range(4):
        st = W.bumpy_config(n, phi, seed=seed, n_small=n_small, n_large=n_large)
        got = []
        for be in (None, oracle()):
            s = W.make_bumpy_system(P.System, st, backend=be, e_c=W.bumpy_contact_scale(st),
                                    method=P.NBR_VERLET)
            out = rows(s)
            s.zero_forces()
            s.compute_forces()
            out += [s.download(f) for f in (P.F_FX, P.F_FY, P.F_TORQUE, P.F_PE)]
            r = s.minimize_fire(spec())
            out += [r.steps, r.avg_pe, s.download(P.F_X), s.download(P.F_ANGLE)] + rows(s)
            got.append(out)
            s.close()
        for a, b in zip(*got):
            assert np.array_equal(a, b), seed


def test_batch_and_server():
    sts = [W.bumpy_config(n, phi, seed=7 * n) for n, phi in SYSTEMS]
    ref = []
    for st in sts:
        s = W.make_bumpy_system(P.System, st, backend=oracle(), e_c=W.bumpy_contact_scale(st),
                                method=P.NBR_VERLET)
        s.minimize_fire(spec())
        ref.append((s.download(P.F_X), s.download(P.F_Y)))
        s.close()
    print("[gpu-case] tiny boxes, batch", len(sts), flush=True)
    b = P.Batch([t.n for t in sts], [t.nv for t in sts])
    for k, t in enumerate(sts):
        b.set_rigid_system(k, t.x, t.y, t.rad, t.mass, t.angle, t.nverts, t.rv, t.side,
                           e_c=W.bumpy_contact_scale(t))
    b.minimize(spec())
    got = [b.get_rigid_system(k)[:2] for k in range(len(sts))]
    b.close()
    print("[gpu-case] tiny boxes, server", len(sts), flush=True)
    sv = P.Server(max_systems=32, arena_slots=1 << 12, budget_bytes=1 << 28,
                  vertex_slots=1 << 14)
    ids = [sv.submit(t.x, t.y, t.rad, t.mass, t.side, P.jam_params(fire=spec()),
                     e_c=W.bumpy_contact_scale(t), angle=t.angle,
                     vertices_per_particle=t.nverts, vertex_radius=t.rv, mode=P.REQ_MINIMIZE)
           for t in sts]
    while any(sv.progress(32)[1:]):
        pass
    served = [sv.result(i) for i in ids]
    for k in range(len(sts)):
        for a, b_, c in zip(ref[k], got[k], (served[k]["x"], served[k]["y"])):
            assert np.array_equal(a, b_), SYSTEMS[k]
            assert np.array_equal(a, c), SYSTEMS[k]
