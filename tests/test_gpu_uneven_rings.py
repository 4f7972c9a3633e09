"""GPU test of rigid particles whose uploaded vertices are unevenly spaced on their rings, off them,
or in another periodic image than their centres: vertex rows entry by entry in row order, forces
and a minimisation from a snapshot, against the oracle bit for bit."""
import numpy as np
import pytest

from _helpers import oracle, pkg, workloads

P = pkg()
W = workloads()
pytestmark = pytest.mark.gpu


def rows(s):
    i, j = s.vertex_pairs()
    o = np.argsort(i, kind="stable")
    return [i[o], j[o]]


def place(st, how):
    """Vertices in static order, spread unevenly on (or off) the rings of st."""
    own = np.repeat(np.arange(st.n), st.nverts)
    k = np.arange(st.nv) - (np.cumsum(st.nverts) - st.nverts)[own]
    t = 2 * np.pi * k / st.nverts[own]
    if how != "even wrapped":
        t = t + 0.3 * np.sin(t)
    r = (st.rad - st.rv)[own] * (1.0 + (0.03 * np.cos(3 * t) if how == "off" else 0.0))
    x, y = (st.x[own] + r * np.cos(t + st.angle[own]), st.y[own] + r * np.sin(t + st.angle[own]))
    if "wrapped" in how:
        x, y = x % st.side, y % st.side
    return x, y


@pytest.mark.parametrize("how", ("uneven", "off", "uneven wrapped", "even wrapped"))
@pytest.mark.parametrize("n,method", ((3, 2), (24, 3), (151, 3), (700, 2), (9001, 3)))
def test_rows_and_minimisation(how, n, method):
    print("[gpu-case] uneven rings", how, n, method, flush=True)
    st = W.bumpy_config(n, 0.86, seed=n, n_small=20, n_large=28 if n != 151 else 40)
    got = []
    for be in (None, oracle()):
        s = W.make_bumpy_system(P.System, st, backend=be, e_c=W.bumpy_contact_scale(st),
                                method=method)
        x, y = place(st, how)
        s.upload(P.F_VERTEX_X, x)
        s.upload(P.F_VERTEX_Y, y)
        s.neighbor_init()
        out = rows(s)
        s.zero_forces()
        s.compute_forces()
        out += [s.download(f) for f in (P.F_FX, P.F_FY, P.F_TORQUE, P.F_PE)]
        s.snapshot_save()
        for _ in range(2):
            r = s.minimize_fire(P.fire_params(avg_pe_target=0.0, avg_pe_diff_target=0.0,
                                              fmax_target=0.0, max_steps=30))
            out += [r.steps, r.avg_pe, s.download(P.F_X), s.download(P.F_ANGLE)] + rows(s)
            s.snapshot_restore()
        got.append(out)
        s.close()
    assert len(got[0][0]) > 0
    for a, b in zip(*got):
        assert np.array_equal(a, b)
