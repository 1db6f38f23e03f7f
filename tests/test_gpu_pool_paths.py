"""Each way a pool steps its systems, asked for by name and seen to have run: the
chunk kernel (packed and not, all pairs, with systems that fault), the per-step
launches, both side by side, and the tuner that chooses between them. FP64
against the oracle or one path against the other, bit for bit."""
import numpy as np
import pytest

import _oracle as O
import _scenarios as S
from test_gpu_pool import agg_case, nl_params, oracle_nl, same
from test_gpu_pool_faults import overflowing

pytestmark = pytest.mark.gpu

R = O.R_PART
DT = 1e-13
CAPACITY, NUMERIC = 5, 4


def pool_of(params, cases, wide_min=None, **kw):
    import libgran_amd as L
    pool = L.Pool(params, max_particles=sum(len(x) for x, _ in cases) + 5000, max_systems=len(cases) + 8, **kw)
    if wide_min is not None:
        pool.set_wide_threshold(wide_min)
        pool.set_split_estimate(False)
    return pool, [pool.add(x, v) for x, v in cases]


def ran(pool, chunk, wide):
    p = pool.last_step_profile()
    assert (p["chunks"] > 0) == chunk and (p["wide_launches"] > 0) == wide, p


@pytest.mark.parametrize("shape", [(512, 1), (256, 2), (256, 8)])
@pytest.mark.parametrize("precision", [0, 1])
def test_packs_in_the_chunk_kernel(precision, shape):
    """Packed and unpacked small systems in the chunk kernel equal the per-step
    launches; FP64 two of them equal the oracle."""
    print(f"[paths] packs, precision {precision}, shape {shape}", flush=True)
    cases = [agg_case(n, 70 + k) for k, n in enumerate((50, 64, 90, 120, 150, 200, 260, 333, 75, 410, 50, 51, 52, 53, 54))]
    wide, ws = pool_of(nl_params(precision), cases, 1)
    wide.step(DT, 120, rebuild_every=50)
    ran(wide, False, True)
    for packing in (True, False):
        pool, slots = pool_of(nl_params(precision), cases, 0)
        pool.set_chunk_shape(*shape)
        pool.set_packing(packing)
        pool.step(DT, 120, rebuild_every=50)
        ran(pool, True, False)
        for a, b in zip(ws, slots):
            same(wide.state(a), pool.state(b), f"packing {packing}")
        if precision == 0:
            for k in (0, 9):
                o = oracle_nl(*cases[k])
                o.step(DT, 120, rebuild_every=50)
                same(o.state(), pool.state(slots[k]), f"oracle, packing {packing}")


@pytest.mark.parametrize("cus", [0, 64])
@pytest.mark.parametrize("precision", [0, 1])
def test_an_exact_threshold_splits_there(precision, cus):
    """Without the estimate the threshold alone decides: 1,500 particles stay in
    the chunk kernel while 4,000 go wide, after one another and side by side."""
    print(f"[paths] exact split, precision {precision}, cus {cus}", flush=True)
    cases = [agg_case(n, 20 + k) for k, n in enumerate((4000, 1500, 300, 90))]
    out = []
    for wide_min in (0, 1, 1501, 4000, 4001):
        pool, slots = pool_of(nl_params(precision), cases, wide_min)
        pool.set_wide_cus(cus)
        pool.step(DT, 130, rebuild_every=50)
        ran(pool, wide_min != 1, 0 < wide_min <= 4000)
        assert pool.split() == dict(wide_from={0: 0, 1: 90, 4001: 0}.get(wide_min, 4000), estimate=False)
        out.append([pool.state(s) for s in slots])
    for other in out[1:]:
        for a, b in zip(out[0], other):
            same(a, b, "split")
    pool, _ = pool_of(nl_params(precision), cases)
    pool.step(DT, 20, rebuild_every=50)
    assert pool.split() == dict(wide_from=90, estimate=True)  # few systems: all wide


def test_the_tuner_tries_splits_and_starts_when_there_is_something_to_tune():
    """A pool that goes wide as a whole counts as tuned; a system that does not
    starts the tuner. It times two shapes, three ways to run the split and the
    thresholds up to the largest system, two intervals each, and results do not
    depend on it."""
    print("[paths] tuner", flush=True)
    cases = [agg_case(n, 90 + k) for k, n in enumerate((3000, 1300, 2200))]
    small = [agg_case(n, 95 + k) for k, n in enumerate((150, 90))]
    outs = []
    for tune in (False, True):
        pool, slots = pool_of(nl_params(1), cases, 1000)
        pool.autotune(tune)
        pool.step(DT, 100, rebuild_every=50)
        ran(pool, False, True)
        assert pool.tuning()["tuned"] == tune
        slots += [pool.add(x, v) for x, v in small]
        pool.step(DT, 100, rebuild_every=50)
        ran(pool, True, True)
        assert not pool.tuning()["tuned"]
        seen, intervals = set(), 2
        while tune and not pool.tuning()["tuned"]:
            pool.step(DT, 50, rebuild_every=50)
            intervals += 1
            seen.add(pool.split()["wide_from"])
            assert intervals < 40
        if tune:
            assert intervals == 2 * (2 + 3 + 3)  # shapes, the split, thresholds of 0, 1024 and 2048
            assert {0, 1300, 2200} <= seen
        pool.step(DT, 50 * (20 - intervals), rebuild_every=50)
        outs.append([pool.state(s) for s in slots])
        pool.autotune(tune)  # from the caller's split again
        pool.step(DT, 50, rebuild_every=50)
        if tune:
            assert pool.split()["wide_from"] == 1300
    for a, b in zip(*outs):
        same(a, b, "tuned")


def test_a_threshold_set_after_tuning_is_the_callers():
    """Whatever the tuner chose, a threshold set later comes with the caller's
    own choice of the estimate, and the estimate with the caller's threshold."""
    print("[paths] after tuning", flush=True)
    cases = [agg_case(n, 90 + k) for k, n in enumerate((3000, 1300, 150))]
    for estimate in (False, True):
        pool, slots = pool_of(nl_params(1), cases)
        pool.set_wide_threshold(2000)
        pool.set_split_estimate(False)  # something narrow to tune
        pool.autotune(True)
        while not pool.tuning()["tuned"] or pool.info(slots[0])[2] == 0:
            pool.step(DT, 50, rebuild_every=50)
        if estimate:
            pool.set_split_estimate(True)
            assert pool.tuning()["wide_min"] == 2000
        pool.set_wide_threshold(1000)
        pool.step(DT, 50, rebuild_every=50)
        assert pool.split() == dict(wide_from=150 if estimate else 1300, estimate=estimate)


def test_all_pairs_lattices_in_the_chunk_kernel():
    print("[paths] all pairs", flush=True)
    import libgran_amd as L
    x, v = S.lattice_with_impactor()
    v2 = v.copy()
    v2[-1] = [0.0, 2.0, -20.0]
    ham = O.hamaker_params(A=1e-20, h0=1e-9)
    p = L.make_params(L.BINARY_CONTACT, L.HAMAKER_FULL, contact=O.contact_params(), hamaker=ham)
    pool, slots = pool_of(p, [(x, v), (x, v2)], 0)
    pool.step(DT, 6000)
    ran(pool, True, False)
    for vv, slot in zip((v, v2), slots):
        o = O.OracleSystem(O.system_params(O.BIN_CONTACT, O.HAM_FULL, hamaker=ham), x, vv)
        o.step(DT, 6000)
        same(o.state(), pool.state(slot), "lattice")
        assert len(o.springs(0)[0]) > 0


@pytest.mark.parametrize("wide_min", [0, 1, 1000])
@pytest.mark.parametrize("precision", [0, 1])
def test_a_lost_system_stops_alone_on_every_path(precision, wide_min):
    print(f"[paths] lost system, precision {precision}, threshold {wide_min}", flush=True)
    import libgran_amd as L
    cases = [agg_case(150, 51), overflowing(200, 54), agg_case(900, 52), agg_case(2500, 53), overflowing(1100, 55)]
    pool, slots = pool_of(nl_params(precision), cases, wide_min)
    with pytest.raises(L.HipgranError) as e:
        pool.step(DT, 120, rebuild_every=50)
    assert e.value.status == NUMERIC
    ran(pool, wide_min != 1, wide_min != 0)
    for k, s in enumerate(slots):
        lost = k in (1, 4)
        assert bool(pool.fault(s)) == lost and pool.info(s)[2] == (50 if lost else 120)
        if not lost:
            q, (t,) = pool_of(nl_params(precision), [cases[k]], 1)
            q.step(DT, 120, rebuild_every=50)
            same(q.state(t), pool.state(s), f"system {k}")


@pytest.mark.parametrize("pairs", [0, 1])
@pytest.mark.parametrize("wide_min", [0, 1])
def test_a_full_table_stops_one_system_on_every_path(wide_min, pairs):
    """A table of two entries: an overlapping lattice needs six."""
    print(f"[paths] full table, threshold {wide_min}, pairs {pairs}", flush=True)
    import libgran_amd as L
    ham = O.hamaker_params(A=1e-20, h0=1e-9)
    kw = dict(pair_mode=1, r_verlet=3.2 * R) if pairs else {}
    p = L.make_params(L.BINARY_CONTACT, L.HAMAKER_FULL, contact=O.contact_params(), hamaker=ham, pair_capacity=2, **kw)
    g = np.stack(np.meshgrid(*[np.arange(3)] * 3, indexing="ij"), axis=-1).reshape(-1, 3) * 1.98 * R
    two = np.array([[0.0, 0.0, 0.0], [2.05 * R, 0.0, 0.0]])
    vv = np.array([[3.0, 0.0, 0.0], [-3.0, 0.0, 0.0]])
    pool, slots = pool_of(p, [(two, vv), (g, np.zeros_like(g)), (two, 2.0 * vv)], wide_min)
    with pytest.raises(L.HipgranError) as e:
        pool.step(DT, 300, rebuild_every=50)
    assert e.value.status == CAPACITY
    ran(pool, wide_min == 0, wide_min == 1)
    assert [bool(pool.fault(s)) for s in slots] == [False, True, False]
    for s, scale in ((slots[0], 1.0), (slots[2], 2.0)):
        o = O.OracleSystem(O.system_params(O.BIN_CONTACT, O.HAM_FULL, neighbor_mode=pairs, hamaker=ham,
                                           **({"r_verlet": 3.2 * R} if pairs else {})), two, scale * vv)
        o.step(DT, 300, rebuild_every=50 * pairs)
        same(o.state(), pool.state(s), "beside it")
