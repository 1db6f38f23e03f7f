"""The per-step tile kernel against the CPU oracle at the edges of its tiles
(64 listed particles, one with all pairs), with lists longer than the 12
positions it handles at once (1,024 with all pairs) and contacts that begin and
end. FP64, so state
and springs must be equal to the last bit."""
import numpy as np
import pytest

import _oracle as O

pytestmark = pytest.mark.gpu

R = O.R_PART


def hot_cloud(n, seed):
    """n spheres near the sites of a touching cubic lattice, some overlapping,
    with velocities that open and close contacts within a few hundred steps."""
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1.0 / 3.0)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), axis=-1).reshape(-1, 3)[:n]
    x = g * 2.0 * R + rng.normal(0.0, 0.004 * R, (n, 3))
    return x, rng.normal(0.0, 10.0, (n, 3)), rng.normal(0.0, 1e8, (n, 3))


@pytest.mark.parametrize("pairs", ["all", "list"])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 63, 64, 65, 129, 257, 1024, 1025, 1026])
def test_tiles_equal_oracle(n, pairs):
    import libgran_amd as L
    print(f"[tile] n {n}, pairs {pairs}", flush=True)
    x, v, w = hot_cloud(n, n)
    kw = dict(r_verlet=5.0 * R) if pairs == "list" else {}
    mode = 1 if pairs == "list" else 0
    ham = O.hamaker_params(A=1e-20, h0=1e-9)
    o = O.OracleSystem(O.system_params(O.BIN_CONTACT, O.HAM_FULL, neighbor_mode=mode, contact=O.contact_params(),
                                       hamaker=ham, **kw), x, v, w0=w)
    s = L.System(L.make_params(L.BINARY_CONTACT, L.HAMAKER_FULL, pair_mode=mode, contact=O.contact_params(),
                               hamaker=ham, **kw), x, v, omega0=w)
    s.per_step_launches(True)
    every = 20 if pairs == "list" else 0
    changed = 0
    last = None
    for steps in (1, 2, 97, 60) if n < 1000 else (1, 2, 7, 20):  # odd and even intervals: both buffers hold the last input
        o.step(1e-13, steps, rebuild_every=every)
        s.step(1e-13, steps, rebuild_every=every)
        a, b = o.state(), s.state()
        for k in ("x", "v", "theta", "omega", "a", "alpha"):
            np.testing.assert_array_equal(b[k], a[k], err_msg=f"{k} after {steps}")
        (ij1, s1), (ij2, s2) = o.springs(0), s.springs(0)
        np.testing.assert_array_equal(ij2, ij1)
        np.testing.assert_array_equal(s2, s1)
        changed += last is not None and (len(last) != len(ij1) or not np.array_equal(last, ij1))
        last = ij1
    if 63 <= n < 1000:
        assert changed  # contacts began or ended between the looks
    s.close()


@pytest.mark.parametrize("terms", ["both", "contact", "hamaker"])
@pytest.mark.parametrize("pairs", [0, 1])
@pytest.mark.parametrize("nf", [1, 4, 5, 9])
def test_facet_terms_in_fours(nf, pairs, terms):
    """Facets four at a time over the threads of a tile: the right fold over
    all of them, in tiles of both kinds."""
    import libgran_amd as L
    from libgran_amd import workloads
    import _scenarios as S
    print(f"[tile] {nf} facets, pairs {pairs}, {terms}", flush=True)
    x = L.generate_aggregate(70, R, 1.8, 1.3, 3)
    v = np.random.default_rng(3).normal(0.0, 1.0, x.shape)
    c, sn, h = S.aggregate_params()
    sets = [workloads.plates(x, R, 5.0 + 0.5 * q) for q in range(3)]
    verts = np.concatenate([q[0] for q in sets])[:nf]
    vel = np.concatenate([q[1] for q in sets])[:nf]
    fac = dict(facet_contact=int(terms != "hamaker"), facet_hamaker=int(terms != "contact"), surface_contact=c,
               surface_hamaker=h)
    kw = dict(r_verlet=3.2 * R) if pairs else {}
    o = O.OracleSystem(O.system_params(O.BIN_SINTER, O.HAM_LIMITED, neighbor_mode=pairs, contact=c, sinter=sn,
                                       hamaker=h, **kw, **fac), x, v)
    s = L.System(L.make_params(L.BINARY_SINTER, L.HAMAKER_LIMITED, pair_mode=pairs, contact=c, sinter=sn, hamaker=h,
                               **kw, **fac), x, v)
    s.per_step_launches(True)
    o.set_facets(verts, vel)
    s.set_facets(verts, vel)
    o.step(1e-13, 60, rebuild_every=20 * pairs)
    s.step(1e-13, 60, rebuild_every=20 * pairs)
    a, b = o.state(), s.state()
    for k in ("x", "v", "theta", "omega", "a", "alpha"):
        np.testing.assert_array_equal(b[k], a[k], err_msg=k)
    s.close()


@pytest.mark.parametrize("steps", [1, 2, 3, 50])
def test_facets_move_with_the_tiles(steps):
    """Two moving facets over tiles of a bonded aggregate: the facets
    alternate between two sets, in odd and even intervals."""
    import libgran_amd as L
    from libgran_amd import workloads
    import _scenarios as S
    print(f"[tile] facets, {steps} steps", flush=True)
    x = L.generate_aggregate(150, R, 1.8, 1.3, 3)
    v = np.random.default_rng(3).normal(0.0, 1.0, x.shape)
    c, sn, h = S.aggregate_params()
    verts, vel = workloads.plates(x, R, 5.0)
    fac = dict(facet_contact=1, facet_hamaker=1, surface_contact=c, surface_hamaker=h)
    o = O.OracleSystem(O.system_params(O.BIN_SINTER, O.HAM_LIMITED, neighbor_mode=1, r_verlet=3.2 * R, contact=c,
                                       sinter=sn, hamaker=h, **fac), x, v)
    s = L.System(L.make_params(L.BINARY_SINTER, L.HAMAKER_LIMITED, pair_mode=1, r_verlet=3.2 * R, contact=c, sinter=sn,
                               hamaker=h, **fac), x, v)
    s.per_step_launches(True)
    o.set_facets(verts, vel)
    s.set_facets(verts, vel)
    for _ in range(2):
        o.step(1e-13, steps, rebuild_every=50)
        s.step(1e-13, steps, rebuild_every=50)
    a, b = o.state(), s.state()
    for k in ("x", "v", "theta", "omega", "a", "alpha"):
        np.testing.assert_array_equal(b[k], a[k], err_msg=k)
    s.close()


@pytest.mark.parametrize("capacity", [2, 3, 4])
@pytest.mark.parametrize("n", [2, 65])
def test_tables_narrower_than_the_tags_read_ahead(n, capacity):
    """A bonded chain whose table and list hold fewer entries than a tile loads
    ahead of their counts."""
    import libgran_amd as L
    import _scenarios as S
    print(f"[tile] chain of {n}, table of {capacity}", flush=True)
    x = np.zeros((n, 3))
    x[:, 0] = 2.0 * R * np.arange(n)
    v = np.random.default_rng(n).normal(0.0, 1.0, x.shape)
    c, sn, h = S.aggregate_params()
    o = O.OracleSystem(O.system_params(O.BIN_SINTER, O.HAM_LIMITED, neighbor_mode=1, r_verlet=3.2 * R, contact=c,
                                       sinter=sn, hamaker=h), x, v)
    s = L.System(L.make_params(L.BINARY_SINTER, L.HAMAKER_LIMITED, pair_mode=1, r_verlet=3.2 * R, contact=c, sinter=sn,
                               hamaker=h, pair_capacity=capacity, neighbor_capacity=2), x, v)
    s.per_step_launches(True)
    for steps in (1, 50):
        o.step(1e-13, steps, rebuild_every=50)
        s.step(1e-13, steps, rebuild_every=50)
    a, b = o.state(), s.state()
    for k in ("x", "v", "theta", "omega", "a", "alpha"):
        np.testing.assert_array_equal(b[k], a[k], err_msg=k)
    s.close()
