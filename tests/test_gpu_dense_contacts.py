"""Beds of touching, unbonded spheres under neighbour lists: every particle has
up to twelve contacts, many of which begin or end in one step, so that a tile
holds more touching pairs than it has threads. FP64: equal to the oracle to the
last bit, in a System and in a Pool over tiles and in the chunk kernel; mixed:
the tiles equal the chunk kernel."""
import numpy as np
import pytest

import _oracle as O

pytestmark = pytest.mark.gpu

R = O.R_PART
TILE, DEPTH, THREADS = 64, 12, 256  # particles, list positions at a time, threads of a tile


def bed(n, seed):
    """n spheres around the sites of a touching face-centred cubic lattice,
    layer by layer, drawn together while they shake."""
    rng = np.random.default_rng(seed)
    m = int(np.ceil((n / 4.0) ** (1.0 / 3.0)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), axis=-1).reshape(-1, 3)
    sites = (g[:, None, :] + np.array([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]])).reshape(-1, 3)[:n]
    x = sites * 2.0 * np.sqrt(2.0) * R + rng.normal(0.0, 0.003 * R, (n, 3))
    return x, rng.normal(0.0, 100.0, (n, 3)) - 1e9 * (x - x.mean(axis=0)), rng.normal(0.0, 1e8, (n, 3))


def touching_in_a_pass(x, offsets, ids):
    """The most touching pairs that one tile has among the list positions it
    takes at a time."""
    n = len(x)
    most = {}
    for i in range(n):
        for k, j in enumerate(ids[offsets[i]:offsets[i + 1]]):
            if np.linalg.norm(x[i] - x[int(j)]) < 2.0 * R:
                key = (i // TILE, k // DEPTH)
                most[key] = most.get(key, 0) + 1
    return max(most.values())


def params(precision, r_list):
    import libgran_amd as L
    return L.make_params(L.BINARY_CONTACT, L.HAMAKER_FULL, pair_mode=1, r_verlet=r_list * R,
                         contact=O.contact_params(), hamaker=O.hamaker_params(A=1e-20, h0=1e-9), precision=precision)


def equal(a, b, what):
    for k in ("x", "v", "theta", "omega", "a", "alpha"):
        np.testing.assert_array_equal(b[k], a[k], err_msg=f"{what}: {k}")


@pytest.mark.parametrize("r_list", [2.2, 2.6, 3.2])
@pytest.mark.parametrize("n", [500, 777])
def test_beds_equal_oracle(n, r_list):
    import libgran_amd as L
    print(f"[bed] n {n}, list {r_list} r", flush=True)
    x, v, w = bed(n, n)
    o = O.OracleSystem(O.system_params(O.BIN_CONTACT, O.HAM_FULL, neighbor_mode=1, r_verlet=r_list * R,
                                       contact=O.contact_params(), hamaker=O.hamaker_params(A=1e-20, h0=1e-9)), x, v, w0=w)
    o.rebuild()
    assert touching_in_a_pass(x, *o.neighbors()) > THREADS
    s = L.System(params(0, r_list), x, v, omega0=w)
    pools = []
    for wide_min in (1, 0):  # tiles, chunk kernel
        pool = L.Pool(params(0, r_list), max_particles=1024, max_systems=2)
        pool.set_wide_threshold(wide_min)
        pools.append((pool, pool.add(x, v, omega0=w)))
    last, both = set(), 0
    for steps in (1, 14, 25, 20, 20):
        for _ in range(steps):
            o.step(1e-13, 1, rebuild_every=20)
            now = set(map(tuple, o.springs(0)[0].tolist()))
            both += len({i for i, _ in now - last} & {i for i, _ in last - now})
            last = now
        s.step(1e-13, steps, rebuild_every=20)
        ij, sp = o.springs(0)
        equal(o.state(), s.state(), f"system after {steps}")
        got = s.springs(0)
        np.testing.assert_array_equal(got[0], ij)
        np.testing.assert_array_equal(got[1], sp)
        for pool, slot in pools:
            pool.step(1e-13, steps, rebuild_every=20)
            equal(o.state(), pool.state(slot), f"pool after {steps}")
            got = pool.springs(slot, 0)
            np.testing.assert_array_equal(got[0], ij)
            np.testing.assert_array_equal(got[1], sp)
    assert both > 100  # a contact began and another ended at one particle in one step
    s.close()
    for pool, _ in pools:
        pool.close()


def test_mixed_beds_in_tiles_equal_the_chunk_kernel():
    import libgran_amd as L
    print("[bed] mixed", flush=True)
    x, v, w = bed(777, 3)
    out = []
    for wide_min in (1, 0):
        pool = L.Pool(params(1, 2.6), max_particles=1024, max_systems=2)
        pool.set_wide_threshold(wide_min)
        slot = pool.add(x, v, omega0=w)
        pool.step(1e-13, 80, rebuild_every=20)
        out.append((pool.state(slot), pool.springs(slot, 0)))
        pool.close()
    equal(out[1][0], out[0][0], "mixed")
    np.testing.assert_array_equal(out[0][1][0], out[1][1][0])
    np.testing.assert_array_equal(out[0][1][1], out[1][1][1])


@pytest.mark.parametrize("first", ["begins", "ends"])
def test_a_full_row_takes_one_contact_for_another(first):
    """A table of one slot: in the step in which one contact of a particle ends
    another begins. The two partners stand in different parts of a list longer
    than a tile takes at a time, in either order."""
    import libgran_amd as L
    print(f"[bed] full row, {first} first", flush=True)
    # particle `mid` between a partner that it leaves and one that comes; 16
    # more within its list, none touching
    k = np.arange(16) + 0.5
    polar, turn = np.arccos(1.0 - 2.0 * k / 16), np.pi * (1.0 + np.sqrt(5.0)) * k
    shell = 4.4 * R * np.stack([np.cos(turn) * np.sin(polar), np.sin(turn) * np.sin(polar), np.cos(polar)], axis=1)
    shell = shell[np.abs(shell[:, 0]) < 3.9 * R]
    assert len(shell) >= 12

    def run(gap):
        come, leave = [[2.0 * R + gap, 0.0, 0.0]], [[-2.0 * R * 0.999, 0.0, 0.0]]
        ends = (come, leave) if first == "begins" else (leave, come)
        x = np.concatenate([ends[0], [[0.0, 0.0, 0.0]], shell, ends[1]])
        v = np.zeros_like(x)
        c, q = (0, len(x) - 1) if first == "begins" else (len(x) - 1, 0)
        v[c, 0] = -20.0
        o = O.OracleSystem(O.system_params(O.BIN_CONTACT, O.HAM_NONE, neighbor_mode=1, r_verlet=5.0 * R,
                                           contact=O.contact_params()), x, v)
        held = []
        for _ in range(60):
            o.step(1e-13, 1)
            ij = o.springs(0)[0]
            held.append(sorted(int(j) for i, j in ij if i == 1))
        return x, v, o, held, c, q

    for gap in np.arange(0.0, 120e-12, 0.25e-12):
        x, v, o, held, c, q = run(gap)
        if any(held[s] == [q] and held[s + 1] == [c] for s in range(59)):
            break
    else:
        raise AssertionError("no gap gives both in one step")
    assert all(len(h) <= 1 for h in held)
    s = L.System(L.make_params(L.BINARY_CONTACT, L.HAMAKER_NONE, pair_mode=1, r_verlet=5.0 * R,
                               contact=O.contact_params(), pair_capacity=1), x, v)
    s.per_step_launches(True)
    s.step(1e-13, 60)
    equal(o.state(), s.state(), first)
    np.testing.assert_array_equal(s.springs(0)[0], o.springs(0)[0])
    np.testing.assert_array_equal(s.springs(0)[1], o.springs(0)[1])
    s.close()


@pytest.mark.parametrize("pairs", [0, 1])
@pytest.mark.parametrize("n", [70, 130])
def test_rows_of_more_than_31_entries(n, pairs):
    """A cloud of spheres pressed into one another that flies apart: rows of
    dozens of entries that end here and there, looked at after every few steps
    and after many."""
    import libgran_amd as L
    print(f"[bed] long rows, n {n}, pairs {pairs}", flush=True)
    rng = np.random.default_rng(n)
    x = rng.uniform(0.0, 2.6 * R, (n, 3))
    v, w = rng.normal(0.0, 300.0, (n, 3)), rng.normal(0.0, 1e8, (n, 3))
    contact = O.contact_params(k=10.0)
    kw = dict(r_verlet=6.0 * R) if pairs else {}
    o = O.OracleSystem(O.system_params(O.BIN_CONTACT, O.HAM_NONE, neighbor_mode=pairs, contact=contact, **kw), x, v, w0=w)
    s = L.System(L.make_params(L.BINARY_CONTACT, L.HAMAKER_NONE, pair_mode=pairs, contact=contact, pair_capacity=n,
                               neighbor_capacity=n if pairs else 0, **kw), x, v, omega0=w)
    s.per_step_launches(True)
    rows = []
    for steps in (1, 2, 5, 40, 40, 80, 80):
        o.step(1e-13, steps, rebuild_every=20)
        s.step(1e-13, steps, rebuild_every=20)
        equal(o.state(), s.state(), f"after {steps}")
        ij = o.springs(0)[0]
        np.testing.assert_array_equal(s.springs(0)[0], ij)
        np.testing.assert_array_equal(s.springs(0)[1], o.springs(0)[1])
        rows.append(np.bincount(ij[:, 0], minlength=n))
    assert rows[-1].max() > 40 and rows[0].sum() - rows[-1].sum() > 50
    s.close()


@pytest.mark.parametrize("n", [32768, 32769])
def test_large_beds_equal_the_tracked_walk(n):
    """512 tiles and one more, from where FP64 tiles run three to a CU;
    dissipation tracking walks."""
    import libgran_amd as L
    print(f"[bed] n {n}", flush=True)
    x, v, w = bed(n, 1)
    out = []
    for tracked in (True, False):
        s = L.System(params(0, 2.6), x, v, omega0=w)
        s.track_dissipation(tracked)
        for steps in (1, 20, 12):
            s.step(1e-13, steps, rebuild_every=20)
        out.append((s.state(), s.springs(0)))
        s.close()
    equal(out[0][0], out[1][0], "tiles")
    np.testing.assert_array_equal(out[1][1][0], out[0][1][0])
    np.testing.assert_array_equal(out[1][1][1], out[0][1][1])


def test_many_aggregates_in_tiles_equal_the_chunk_kernel():
    """70 aggregates of 500 in 560 tiles."""
    import libgran_amd as L
    import _scenarios as S
    print("[bed] 560 tiles of aggregates", flush=True)
    c, sn, h = S.aggregate_params()
    p = L.make_params(L.BINARY_SINTER, L.HAMAKER_LIMITED, pair_mode=1, r_verlet=3.2 * R, contact=c, sinter=sn, hamaker=h)
    cases = [L.generate_aggregate(500, R, 1.8, 1.3, k) for k in range(70)]
    out = []
    for wide_min in (1, 0):
        pool = L.Pool(p, max_particles=36000, max_systems=70)
        pool.set_wide_threshold(wide_min)
        slots = [pool.add(x, np.random.default_rng(k).normal(0.0, 1.0, x.shape)) for k, x in enumerate(cases)]
        pool.step(1e-13, 120, rebuild_every=50)
        assert (pool.last_step_profile()["chunks"] == 0) == (wide_min == 1)
        out.append([(pool.state(s), pool.springs(s, 1)) for s in slots])
        pool.close()
    for (a, sa), (b, sb) in zip(*out):
        equal(a, b, "aggregate")
        np.testing.assert_array_equal(sb[1], sa[1])
