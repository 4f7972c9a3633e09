"""GPU test of the rule that sends small disk systems to the one-workgroup loops, around its lines,
against the oracle bit for bit: size classes chosen for the pairs, systems too dense for them,
and clusters in a large box, whose density the rule does not see."""
import numpy as np
import pytest

from _helpers import oracle, pkg, workloads
from test_gpu_resident import fire, heat, same

P = pkg()
W = workloads()
pytestmark = pytest.mark.gpu


def pair(n, phi, method, skin, spread):
    st = W.disk_config(n, phi, seed=n)
    st.side *= spread
    if spread > 1:
        st.x, st.y = st.x + 0.4 * st.side, st.y + 0.3 * st.side
    spec = W.neighbor_spec(st.side, skin=skin, method=method)
    spec.n_cells_dim = min(spec.n_cells_dim, 38)  # (more cells than a class holds chunk the loop)
    return [W.make_disk_system(P.System, st, spec, backend=be) for be in (None, oracle())]


@pytest.mark.parametrize("method", (P.NBR_CELL, P.NBR_VERLET))
@pytest.mark.parametrize("n,phi,skin,spread", (
    (100, 0.84, 1.0, 1), (256, 0.84, 0.6, 1), (256, 0.84, 1.0, 1), (257, 0.84, 1.0, 1),
    (384, 0.84, 0.8, 1), (384, 0.84, 0.95, 1), (500, 0.84, 0.6, 1), (512, 0.95, 0.6, 1),
    (768, 0.84, 1.0, 1), (769, 0.84, 1.0, 1), (1000, 0.84, 0.6, 1), (1024, 0.84, 0.8, 1),
    (1536, 0.84, 0.6, 1), (1700, 0.84, 0.45, 1), (2048, 0.84, 0.3, 1), (2048, 0.84, 0.6, 1),
    (250, 1.5, 0.3, 4), (600, 1.5, 0.3, 4), (1400, 1.5, 0.3, 3), (600, 1.0, 1.2, 4),
))
def test_routes(n, phi, skin, spread, method):
    print("[gpu-case] resident routes", n, phi, skin, spread, method, flush=True)
    g, o = pair(n, phi, method, skin, spread)
    rg, ro = fire(g, 60), fire(o, 60)
    assert (rg.steps, rg.avg_pe, rg.fmax_sq) == (ro.steps, ro.avg_pe, ro.fmax_sq)
    same(g, o, "fire")
    heat((g, o), 1e-2, n)
    for s in (g, o):
        s.nve_run(0.01, 50)
    same(g, o, "nve")


def test_a_wider_skin_changes_the_route_of_a_system():
    """The same system, configured again: each route goes on from the other's state."""
    g, o = pair(1000, 0.84, P.NBR_CELL, 0.3, 1)
    heat((g, o), 1e-2)
    for skin in (0.3, 1.0, 0.6, 0.3):
        for s in (g, o):
            W.configure(s, W.neighbor_spec(s.box()[0], skin=skin))
            s.neighbor_init()
            s.nve_run(0.01, 40)
        same(g, o, skin)
