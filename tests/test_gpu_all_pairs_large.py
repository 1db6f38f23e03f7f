"""All-pairs systems on both sides of the size from which a lane walks a
particle's partners instead of a workgroup: the two give the same bits."""
import numpy as np
import pytest

import _oracle as O
import _scenarios as S
from test_gpu_dense_contacts import bed, equal

pytestmark = pytest.mark.gpu

R = O.R_PART
DT = 1e-13


@pytest.mark.parametrize("n,ham", [(17999, "NONE"), (18001, "NONE"), (30001, "FULL")])
def test_contact_systems_equal_the_tracked_walk(n, ham):
    """Dissipation tracking walks at every size."""
    import libgran_amd as L
    print(f"[all pairs] contact {ham}, n {n}", flush=True)
    x, v, w = bed(n, 1)
    p = L.make_params(L.BINARY_CONTACT, getattr(L, f"HAMAKER_{ham}"), contact=O.contact_params(),
                      hamaker=O.hamaker_params(A=1e-20, h0=1e-9))
    out = []
    for tracked in (True, False):
        s = L.System(p, x, v, omega0=w)
        s.track_dissipation(tracked)
        s.step(DT, 3)
        out.append((s.state(), s.springs(0)))
        s.close()
    equal(out[0][0], out[1][0], ham)
    assert len(out[0][1][0]) > n
    np.testing.assert_array_equal(out[1][1][0], out[0][1][0])
    np.testing.assert_array_equal(out[1][1][1], out[0][1][1])


@pytest.mark.parametrize("binary,n", [("NONE", 18100), ("SINTER", 30100)])
def test_systems_within_a_cutoff_equal_their_lists(binary, n):
    """With an attraction that ends at three radii all pairs and a list of 3.2
    give the same sums."""
    import libgran_amd as L
    print(f"[all pairs] {binary}, n {n}", flush=True)
    x = L.generate_aggregate(n, R, 1.8, 1.3, 2)
    v = np.random.default_rng(2).normal(0.0, 1.0, x.shape)
    c, sn, h = S.aggregate_params()
    out = []
    for kw in ({}, dict(pair_mode=L.PAIRS_NEIGHBOR_LIST, r_verlet=3.2 * R)):
        s = L.System(L.make_params(getattr(L, f"BINARY_{binary}"), L.HAMAKER_LIMITED, contact=c, sinter=sn, hamaker=h,
                                   **kw), x, v)
        s.step(DT, 3)
        out.append(s.state())
        s.close()
    equal(out[0], out[1], binary)
