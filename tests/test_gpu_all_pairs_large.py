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


@pytest.mark.parametrize("precision,ham,n", [(0, "NONE", 18100), (0, "FULL", 30100), (1, "NONE", 20100)])
def test_pools_equal_other_paths(precision, ham, n):
    """A large system and a small one in a pool, in odd and even intervals with
    moving facets: FP64 equals the tracked walk of single systems, mixed the
    chunk kernel."""
    import libgran_amd as L
    print(f"[all pairs] pool {ham}, n {n}, precision {precision}", flush=True)
    c, _, _ = S.aggregate_params()
    p = L.make_params(L.BINARY_CONTACT, getattr(L, f"HAMAKER_{ham}"), contact=O.contact_params(),
                      hamaker=O.hamaker_params(A=1e-20, h0=1e-9), precision=precision, facet_contact=1, facet_hamaker=1,
                      surface_contact=c, surface_hamaker=O.hamaker_params(A=1e-20, h0=1e-10))
    cases = [bed(n, 1), bed(300, 2)]
    from libgran_amd import workloads as W
    plates = W.plates(cases[1][0], R, 6.0)
    pool = L.Pool(p, max_particles=n + 400, max_systems=3, max_facets=4)
    slots = [pool.add(x, v, omega0=w) for x, v, w in cases]
    pool.set_facets(slots[1], *plates)
    for steps in (1, 1, 2, 2, 1):  # a recorded interval is replayed
        pool.step(DT, steps)
    assert pool.last_step_profile()["wide_launches"] == 3
    for k, (x, v, w) in enumerate(cases):
        if precision == 0:
            s = L.System(p, x, v, omega0=w)
            s.track_dissipation(True)
            if k:
                s.set_facets(*plates)
            s.step(DT, 7)
            ref, springs = s.state(), s.springs(0)
        else:
            q = L.Pool(p, max_particles=n + 64, max_systems=1, max_facets=4)
            q.set_wide_threshold(0)
            slot = q.add(x, v, omega0=w)
            if k:
                q.set_facets(slot, *plates)
            q.step(DT, 7)
            ref, springs = q.state(slot), q.springs(slot, 0)
        equal(ref, pool.state(slots[k]), f"system {k}")
        got = pool.springs(slots[k], 0)
        np.testing.assert_array_equal(got[0], springs[0])
        np.testing.assert_array_equal(got[1], springs[1])
