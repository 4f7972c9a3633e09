"""GPU test of the vertex rows (RigidBumpy::updateVertexVerletList) against the oracle, entry
by entry in row order: rings of few, usual and more than 32 vertices, rings so small that every
vertex is a candidate, boxes of a few cells with rows across the edge, and rings that are not
evenly spaced counterclockwise (which take the general build)."""
import numpy as np
import pytest

from _helpers import oracle, pkg, workloads

P = pkg()
W = workloads()
pytestmark = pytest.mark.gpu


def rows(s):
    i, j = s.vertex_pairs()
    o = np.argsort(i, kind="stable")  # each vertex's row, in row order
    return i[o], j[o]



@pytest.mark.parametrize("n_small,n_large", ((3, 5), (7, 12), (20, 28), (33, 40), (9, 64)))
@pytest.mark.parametrize("n,reverse", ((24, False), (151, False), (151, True)))
def test_rows_equal_the_oracle(n_small, n_large, n, reverse):
    print("[gpu-case] vertex rows", n_small, n_large, n, reverse, flush=True)
    st = W.bumpy_config(n, 0.88, seed=n + n_small, n_small=n_small, n_large=n_large)
    got = []
    for be in (None, oracle()):
        s = W.make_bumpy_system(P.System, st, backend=be, e_c=W.bumpy_contact_scale(st))
        if reverse:  # the same rings, numbered clockwise
            first = np.cumsum(st.nverts) - st.nverts
            order = np.concatenate([np.arange(a + k - 1, a - 1, -1)
                                    for a, k in zip(first, st.nverts)])
            for f in (P.F_VERTEX_X, P.F_VERTEX_Y):
                s.upload(f, s.download(f)[order])
            s.neighbor_init()
        a = rows(s)
        s.upload(P.F_OMEGA, np.linspace(-2.0, 2.0, n))
        s.nve_run(0.01, 3)  # turned rings
        s.neighbor_init()
        got.append(a + rows(s))
        s.close()
    for g, o in zip(*got):
        assert np.array_equal(g, o)
    assert len(got[0][0]) > 0
