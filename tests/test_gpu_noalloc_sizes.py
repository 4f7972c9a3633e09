"""GPU test of dpm_disk_forces_noalloc over its branches, against the list-based entry points bit
for bit: chunk edges, both grids (in LDS up to 8,192 particles, in memory beyond), three cells a
side, particles with more pairs than LDS holds, positions outside the box, a general exponent,
radii beyond the short sequences' range, and replays of a captured call."""
import ctypes as C

import numpy as np
import pytest
import torch

from _helpers import pkg, workloads

P = pkg()
W = workloads()
pytestmark = pytest.mark.gpu


def bare(st, cutoff, e_c=1.0, n_c=2.0, graph=False):
    dev = torch.device("cuda")
    x, y, r = (torch.from_numpy(np.ascontiguousarray(a)).to(dev) for a in (st.x, st.y, st.rad))
    fx, fy, pe = (torch.full((st.n,), 7.0, dtype=torch.float64, device=dev) for _ in range(3))
    tot = torch.full((1,), 7.0, dtype=torch.float64, device=dev)

    def call():
        P.load().call("disk_forces_noalloc", x.data_ptr(), y.data_ptr(), r.data_ptr(), st.n,
                      st.side, st.side, e_c, n_c, cutoff, fx.data_ptr(), fy.data_ptr(),
                      pe.data_ptr(), tot.data_ptr(), torch.cuda.current_stream().cuda_stream)

    call()
    torch.cuda.synchronize()
    out = [a.cpu().numpy() for a in (fx, fy, pe, tot)]
    if graph:
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            call()
        for _ in range(3):
            for a in (fx, fy, pe, tot):
                a.fill_(7.0)
            g.replay()
            torch.cuda.synchronize()
            for a, b in zip(out, (fx, fy, pe, tot)):
                assert np.array_equal(a, b.cpu().numpy())
    return out


def listed(st, cutoff, e_c=1.0, n_c=2.0):
    s = W.make_disk_system(P.System, st, W.NeighborSpec(2, cutoff, 3 * 0.15 ** 2, 3, 1e30),
                           e_c=e_c, n_c=n_c)
    s.zero_forces()
    s.compute_forces()
    out = [s.download(P.F_FX), s.download(P.F_FY), s.download(P.F_PE),
           np.array([s.reduce(P.RED_PE)])]
    s.close()
    return out


@pytest.mark.parametrize("n,phi,cutoff,e_c,n_c,scale", (
    (1, 0.05, 1.7, 1.0, 2.0, 1.0),
    (24, 0.9, 1.7, 1.0, 2.0, 1.0),        # three cells a side
    (63, 0.85, 1.7, 1.0, 2.0, 1.0),
    (64, 0.85, 1.7, 1.0, 2.0, 1.0),
    (65, 0.85, 1.7, 1.0, 2.5, 1.0),
    (1500, 0.85, 1.7, 0.3, 2.0, 1.0),
    (1025, 6.0, 1.7, 1.0, 2.0, 1.0),      # some 30 to 70 pairs a particle
    (700, 0.85, 1.7 * 2.0 ** -110, 1.0, 2.0, 2.0 ** -110),
    (8192, 0.86, 1.7, 1.0, 2.0, 1.0),
    (8193, 0.86, 1.7, 1.0, 2.5, 1.0),
    (50021, 0.02, 1.7, 1.0, 2.0, 1.0),    # more cells than the grid may have
    (8001, 0.02, 1.7, 1.0, 2.0, 1.0),
    (40009, 3.0, 2.1, 1.0, 2.0, 1.0),
))
def test_equals_the_list_path(n, phi, cutoff, e_c, n_c, scale):
    print("[gpu-case] noalloc", n, phi, cutoff, e_c, n_c, scale, flush=True)
    st = W.disk_config(n, phi, seed=n)
    rng = np.random.default_rng(n)
    st.x = (st.x + st.side * rng.integers(-2, 3, n)) * scale  # unwrapped coordinates
    st.y = st.y * scale
    st.rad = st.rad * scale
    st.side *= scale
    got, ref = bare(st, cutoff, e_c, n_c, graph=n in (1500, 8193)), listed(st, cutoff, e_c, n_c)
    for k, name in enumerate(("fx", "fy", "pe", "total")):
        assert np.array_equal(got[k], ref[k]), (name, np.max(np.abs(got[k] - ref[k])))
    assert n == 1 or phi < 0.1 or np.max(np.abs(got[0])) > 0
