"""GPU test of the launch that builds a rigid system's particle and vertex rows together, against
the oracle entry by entry in row order: sizes around a block's and the rule's limit, a box of
three cells a side, rows of more entries than its LDS list holds, and the runs that follow."""
import numpy as np
import pytest

from _helpers import oracle, pkg, workloads

P = pkg()
W = workloads()
pytestmark = pytest.mark.gpu


def rows(s):
    out = []
    for i, j in (s.neighbor_pairs(), s.vertex_pairs()):
        o = np.argsort(i, kind="stable")  # each row in row order
        out += [i[o], j[o]]
    return out


@pytest.mark.parametrize("n,phi,cells,verts,steps", (
    (9, 0.5, 3, (20, 28), 40),
    (257, 0.8, 0, (20, 28), 40),
    (60, 6.0, 3, (4, 6), 3),       # every particle a neighbour of nearly every other
    (200, 6.0, 3, (4, 6), 3),      # some 100 entries a row
    (8192, 0.8, 0, (6, 8), 3),
    (8193, 0.8, 0, (6, 8), 3),
))
def test_rows_and_runs_equal_the_oracle(n, phi, cells, verts, steps):
    print("[gpu-case] fused lists", n, phi, cells, verts, steps, flush=True)
    st = W.bumpy_config(n, phi, seed=n, n_small=verts[0], n_large=verts[1])
    got = []
    for be in (None, oracle()):
        s = W.make_bumpy_system(P.System, st, backend=be, e_c=W.bumpy_contact_scale(st))
        first = rows(s)
        s.minimize_fire(P.fire_params(max_steps=steps))
        st_ = s.neighbor_stats()
        got.append((first, rows(s),
                    [s.download(f) for f in (P.F_X, P.F_Y, P.F_ANGLE, P.F_FX, P.F_TORQUE)], st_))
        s.close()
    (g0, g1, gf, gs), (o0, o1, of, os_) = got
    for a, b in zip(g0 + g1 + gf, o0 + o1 + of):
        assert np.array_equal(a, b)
    assert gs == os_
    assert phi < 2 or n < 200 or os_["max_alloc"] > 64
