"""GPU test of the transfers between the caller's arrays (static order) and the device's
(cell order), at sizes on both sides of a workgroup and of the pinned staging buffer (512 KiB:
65,536 values): what was uploaded comes back bit for bit, and reductions read what was
uploaded."""
import numpy as np
import pytest

from _helpers import oracle, pkg, workloads

P = pkg()
W = workloads()
pytestmark = pytest.mark.gpu

FIELDS = (P.F_X, P.F_Y, P.F_VX, P.F_VY, P.F_FX, P.F_FY, P.F_RAD, P.F_MASS, P.F_PE)


@pytest.mark.parametrize("n", (64, 257, 65536, 65537))
def test_fields_return_as_uploaded_in_static_order(n):
    print("[gpu-case] exchange", n, flush=True)
    st = W.disk_config(n, 0.80, seed=n)
    s = W.make_disk_system(P.System, st)  # the cell sort permutes the device's order
    perm = s.download(P.F_STATIC_INDEX)
    assert np.array_equal(np.sort(perm), np.arange(n)) and not np.array_equal(perm, np.arange(n))
    rng = np.random.default_rng(n)
    sent = {f: rng.uniform(0.25, 1.0, n) for f in FIELDS}
    for f, a in sent.items():
        s.upload(f, a)
    for f, a in sent.items():
        assert np.array_equal(s.download(f), a), f
    s.close()


@pytest.mark.parametrize("n", (257, 4097))
def test_reductions_equal_the_oracle(n):
    print("[gpu-case] reductions", n, flush=True)
    st = W.disk_config(n, 0.86, seed=n)
    got = []
    for be in (None, oracle()):
        s = W.make_disk_system(P.System, st, backend=be)
        s.upload(P.F_VX, st.x - st.x.mean())
        s.zero_forces()
        s.compute_forces()
        got.append([s.reduce(q) for q in (P.RED_PE, P.RED_KE, P.RED_POWER, P.RED_FMAX_SQ,
                                          P.RED_FORCE_BALANCE, P.RED_PRESSURE, P.RED_CONTACTS,
                                          P.RED_PACKING_FRACTION)]
                   + [s.download(P.F_NUM_NEIGHBORS).sum(), s.download(P.F_CONTACTS).sum()])
        s.close()
    assert got[0] == got[1]
