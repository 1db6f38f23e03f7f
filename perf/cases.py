"""What a program that uses this framework has it do, as cases that can be timed and compared.

A case is one call pattern on one kind of system:

  system   one aggregate or lattice in a `System`: `steps` velocity-Verlet steps, then the state is read
  ledger   the driver's thermo loop: runs of steps with the momenta, kinetic terms and energy ledger read in between
  pool     many uneven aggregates stepped together in a `Pool`, then every state is read
  serve    plate tests submitted to a `Server`, each waited for and read

Geometry, parameter sets and sizes are those of this repository's benchmark, tests and the scenarios they cite: 14 nm
spheres of 1700 kg/m^3, dt 1e-13 s, touching lattices of a few dozen to a few hundred spheres, cluster-cluster aggregates
of 50 to 20,000, batches with log-normal sizes (median 400).

`exact` steps the same inputs in NumPy, pair by pair in 64 bits, for everything but the facets and the batches.
"""
import math

import numpy as np

import libgran_amd as L
from libgran_amd import workloads

R = 1.4e-8
MASS = 4.0 / 3.0 * math.pi * R ** 3 * 1700.0
INERTIA = 2.0 / 5.0 * MASS * R ** 2
DT = 1e-13
FIELDS = ("x", "v", "theta", "omega", "a", "alpha")


def listed():
    return [
        # A driver of the impact scenario calls one step at a time and looks at the state after each: the smallest call.
        dict(name="impact19_one_step", kind="system", shape="impact", n=19, pairs="all", binary="contact", steps=1),
        # The same scenario under its 5r neighbour list, rebuilt every 20 steps, between two thermo lines.
        dict(name="impact19_list", kind="system", shape="impact", n=19, pairs="list", r_list=5.0, rebuild=20,
             binary="contact", steps=200),
        # The bonded 3x3x3 lattice of the legacy connector model, every pair evaluated.
        dict(name="lattice27_legacy", kind="system", shape="block", n=27, pairs="all", binary="legacy", steps=200),
        # Two lattice balls flying at each other, contact and long-range attraction between all pairs (the demo driver).
        dict(name="collision522_all_pairs", kind="system", shape="balls", n=522, pairs="all", binary="contact", steps=20),
        # One small soot aggregate in double precision, the basic workload of the benchmark.
        dict(name="aggregate200", kind="system", shape="aggregate", n=200, pairs="list", r_list=3.2, rebuild=50,
             binary="sinter", precision="fp64", steps=500),
        # A mid-size aggregate pressed between two moving plates in double precision.
        dict(name="plates1777", kind="system", shape="aggregate", n=1777, pairs="list", r_list=3.2, rebuild=50,
             binary="sinter", precision="fp64", plates=True, steps=100),
        # The large aggregate of the benchmark, in double and in mixed precision.
        dict(name="aggregate20000", kind="system", shape="aggregate", n=20000, pairs="list", r_list=3.2, rebuild=50,
             binary="sinter", precision="fp64", steps=100),
        dict(name="aggregate20000_mixed", kind="system", shape="aggregate", n=20000, pairs="list", r_list=3.2,
             rebuild=50, binary="sinter", precision="mixed", steps=100),
        # A run that logs: ten steps, then diagnostics and the energy ledger, five times.
        dict(name="ledger5000", kind="ledger", shape="aggregate", n=5000, pairs="list", r_list=3.2, rebuild=50,
             binary="sinter", precision="fp64", steps=50, every=10),
        # A batch of uneven aggregates in mixed precision with the settings the benchmark fixes.
        dict(name="batch1024_mixed", kind="pool", systems=1024, median=400, precision="mixed", tuned=True, steps=2000),
        # A smaller batch in double precision with the pool's own defaults.
        dict(name="batch333_fp64", kind="pool", systems=333, median=400, precision="fp64", tuned=False, steps=800),
        # Requests of a serving stream: aggregates between moving plates, submitted together, waited for in turn.
        dict(name="serve24_mixed", kind="serve", requests=24, n_low=100, n_high=6000, precision="mixed", steps=1000),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("scenario", "balls", "aggregate", "aggregate", "aggregate", "ledger", "pool", "serve"))
    listing = dict(pairs="list", r_list=3.2, rebuild=50, binary="sinter")
    if kind == "scenario":
        case = dict(kind="system", steps=_log(rng, 1, 400))
        if rng.random() < 0.3:
            return dict(case, shape="block", n=27, pairs="all", binary="legacy")
        case.update(shape="impact", n=19, binary="contact", pairs="all")
        if rng.random() < 0.5:
            case.update(pairs="list", r_list=5.0, rebuild=20)
        return case
    if kind == "balls":
        return dict(kind="system", shape="balls", n=_log(rng, 40, 700), pairs="all", binary="contact",
                    steps=_log(rng, 4, 20))
    if kind == "aggregate":
        return dict(kind="system", shape="aggregate", n=_log(rng, 50, 20000), **listing,
                    precision=rng.choice(("fp64", "mixed")), plates=rng.random() < 0.25, steps=rng.randint(30, 100))
    if kind == "ledger":
        every = rng.randint(5, 25)
        return dict(kind="ledger", shape="aggregate", n=_log(rng, 100, 8000), **listing,
                    precision=rng.choice(("fp64", "mixed")), steps=every * rng.randint(2, 4), every=every)
    if kind == "pool":
        return dict(kind="pool", systems=_log(rng, 5, 800), median=rng.randint(150, 500),
                    precision=rng.choice(("fp64", "mixed")), tuned=rng.random() < 0.5, steps=rng.randint(100, 600))
    low = rng.randint(80, 300)
    return dict(kind="serve", requests=_log(rng, 3, 20), n_low=low, n_high=low * rng.randint(4, 18),
                precision=rng.choice(("fp64", "mixed")), steps=rng.randint(200, 800))


# ------------------------------------------------------------------ parameters


def _functors(binary):
    """Contact, bond and Hamaker parameter sequences: the lattice scenarios' and the aggregates'."""
    if binary in ("contact", "legacy"):
        k, gn, kb = 1.0e4, 5.0e-9, 1.0e4
        contact = [k, gn, k, 0.2 * gn, 1.0, 1.0, k, 0.05 * gn, 0.1, 1.0, k, 0.05 * gn, 0.1, 1.0, R, MASS, INERTIA, DT]
        return contact, [kb, 0.0, kb, 0.0, kb, 0.0, kb, 0.0, R, MASS, INERTIA, DT, 1.0e-9], [1e-20, 1e-9, 3 * R, R, MASS]
    k = 1.0e4
    g = 2.0 * 0.5 * math.sqrt(k * MASS / 2.0)
    contact = [k, g, k, g, 1.0, 1.0, k, g, 1.0, 1.0, k, g, 1.0, 1.0, R, MASS, INERTIA, DT]
    return contact, [k, g, k, g, k, g, k, g, R, MASS, INERTIA, DT, 1e-3 * R], [1e-20, 1e-10, 3 * R, R, MASS]


def _hamaker(case):
    return {"contact": "full", "legacy": None}.get(case.get("binary", "sinter"), "limited")


def _params(case, facets):
    binary = case.get("binary", "sinter")
    contact, sinter, hamaker = _functors(binary)
    extra = {}
    if case.get("pairs", "list") == "list":
        extra.update(pair_mode=L.PAIRS_NEIGHBOR_LIST, r_verlet=case.get("r_list", 3.2) * R)
    if facets:
        extra.update(facet_contact=1, facet_hamaker=1, surface_contact=contact, surface_hamaker=hamaker)
    return L.make_params({"contact": L.BINARY_CONTACT, "sinter": L.BINARY_SINTER, "legacy": L.BINARY_SINTER_LEGACY}[binary],
                         {None: L.HAMAKER_NONE, "full": L.HAMAKER_FULL, "limited": L.HAMAKER_LIMITED}[_hamaker(case)],
                         contact=contact, sinter=sinter, hamaker=hamaker,
                         precision=L.PRECISION_MIXED if case.get("precision") == "mixed" else L.PRECISION_FP64, **extra)


# ---------------------------------------------------------------------- inputs


def _ball(n):
    """The n sites of a simple cubic lattice of touching spheres nearest to a point off its symmetry axes."""
    m = int(math.ceil(n ** (1.0 / 3.0))) + 2
    g = np.stack(np.meshgrid(*[np.arange(-m, m + 1)] * 3, indexing="ij"), axis=-1).reshape(-1, 3).astype(np.float64)
    d = np.linalg.norm(g - np.array([0.11, 0.07, 0.03]), axis=1)
    return g[np.argsort(d, kind="stable")[:n]] * (2.0 * R)


def _inputs(case, seed):
    """Positions, velocities and angular velocities of one system, from the seed alone."""
    rng = np.random.default_rng(seed)
    n, shape = case["n"], case["shape"]
    if shape == "impact":  # two 3x3 layers at rest and one sphere above them, moving down
        x = [[(-3.0 + 2.0 * j) * R, (-3.0 + 2.0 * i) * R, z] for i in range(3) for j in range(3) for z in (0.0, -2.0 * R)]
        x = np.array(x + [[0.0, 0.0, 3.0 * R]])
        v = rng.normal(0.0, 0.01, x.shape)
        v[-1] += [1.0, 0.0, -10.0]
        return x, v, np.zeros_like(x)
    if shape == "block":  # 3x3x3 touching spheres, two opposite columns pulled in different directions
        x = np.array([[(2.0 * j - 1.0) * R, (2.0 * i - 1.0) * R, -2.0 * k * R]
                      for i in range(3) for j in range(3) for k in range(3)])
        v = rng.normal(0.0, 0.05, x.shape)
        v += np.array([[0.0, 0.0, 5.0] if j == 0 else ([0.0, 5.0, 0.0] if j == 2 else [0.0, 0.0, 0.0])
                       for i in range(3) for j in range(3) for k in range(3)])
        return x, v, np.zeros_like(x)
    if shape == "balls":  # two lattice balls half a radius apart, closing at 4 m/s off their line of centres
        a, b = _ball(n // 2), _ball(n - n // 2)
        b[:, 0] += a[:, 0].max() - b[:, 0].min() + 2.5 * R
        v = rng.normal(0.0, 0.05, (n, 3))
        v[: n // 2] += [2.0, 0.1, 0.0]
        v[n // 2:] -= [2.0, 0.1, 0.0]
        return np.concatenate([a, b]), v, rng.normal(0.0, 1e6, (n, 3))
    x = L.generate_aggregate(n, R, 1.8, 1.3, seed)
    return x, rng.normal(0.0, 1.0, x.shape), np.zeros_like(x)


def _plates(x, seed):
    return workloads.plates(x, R, float(np.random.default_rng(seed + 77).uniform(1.0, 10.0)), True)


def _unit_vectors(seed):
    rng = np.random.default_rng(seed + 5)

    def one():
        q = rng.uniform(-1.0, 1.0, 3)
        return q / np.linalg.norm(q)
    return one


def _batch(case, seed):
    """Aggregates of log-normal sizes, the same sizes for every seed, and their velocities."""
    sizes, dfs = workloads.batch_sizes(case["systems"], median=case["median"], hi=6000, seed=case["systems"])
    rng = np.random.default_rng(seed)
    xs = L.generate_aggregates(sizes, dfs, 1.3, rng.integers(1, 1 << 40, len(sizes), dtype=np.uint64), R)
    return xs, [rng.normal(0.0, 1.0, x.shape) for x in xs]


def _requests(case, seed):
    """Plate tests of log-uniform sizes, the same sizes for every seed: positions and moving plates."""
    sizes = np.random.default_rng(case["requests"]).uniform(math.log(case["n_low"]), math.log(case["n_high"]), case["requests"])
    rng = np.random.default_rng(seed)
    xs = L.generate_aggregates(np.round(np.exp(sizes)).astype(np.uint32), rng.uniform(1.6, 2.2, len(sizes)), 1.3,
                               rng.integers(1, 1 << 40, len(sizes), dtype=np.uint64), R)
    return [dict(x=x, facets=workloads.plates(x, R, rng.uniform(1.0, 10.0), rng.random() < 0.5)) for x in xs]


def prepare(case, seed):
    if case["kind"] == "pool":
        xs, vs = _batch(case, seed)
        pool = L.Pool(_params(case, False), max_particles=sum(len(x) for x in xs) + 1024, max_systems=len(xs))
        if case["tuned"]:
            pool.set_chunk_shape(512, 1)
            pool.set_wide_threshold(4096)
            pool.set_wide_cus(0)
        slots = [pool.add(x, v) for x, v in zip(xs, vs)]
        return dict(case=case, pool=pool, slots=slots)
    if case["kind"] == "serve":
        stream = _requests(case, seed)
        p = _params(case, True)
        room = sum(len(q["x"]) for q in stream) + 4096
        server = L.Server(p, L.Pool.bytes_per_particle(p, 4) * room, case["requests"], max_facets=4, quantum=1000,
                          rebuild_every=50, dt=DT)
        return dict(case=case, server=server, stream=stream)
    x, v, w = _inputs(case, seed)
    system = L.System(_params(case, case.get("plates", False)), x, v, None, w)
    if case.get("plates"):
        system.set_facets(*_plates(x, seed))
    if case["binary"] == "legacy":
        system.set_legacy_connectors(*L.legacy_sinter_frames(x, R, 1.0e-9, _unit_vectors(seed)))
    return dict(case=case, system=system)


# ------------------------------------------------------------------------- run


def _columns(lines):
    """A log's columns: momenta, radius of gyration and the ledger's terms, one array each."""
    return dict(zip(("P", "L", "rg") + L.ENERGY_TERMS, np.array(lines).T.copy()))


def run(state):
    case = state["case"]
    if case["kind"] == "pool":
        pool = state["pool"]
        pool.step(DT, case["steps"], rebuild_every=50)
        got = [pool.state(s) for s in state["slots"]]
        return {f: np.concatenate([g[f] for g in got]) for f in FIELDS}
    if case["kind"] == "serve":
        server = state["server"]
        ids = [server.submit(q["x"], case["steps"], facets=q["facets"]) for q in state["stream"]]
        got = [server.wait(i) for i in ids]
        return {f: np.concatenate([g[f] for g in got]) for f in FIELDS[:4]}
    system = state["system"]
    if case["kind"] == "ledger":
        lines = []
        for _ in range(case["steps"] // case["every"]):
            system.step(DT, case["every"], rebuild_every=case["rebuild"])
            d, e = system.diagnostics(MASS, INERTIA), system.energy(MASS, INERTIA)
            lines.append([d["P"], d["L"], d["rg"]] + [e[t] for t in L.ENERGY_TERMS])
        return dict(system.state(), **_columns(lines))
    system.step(DT, case["steps"], rebuild_every=case.get("rebuild", 0))
    return system.state()


# ------------------------------------------------------------------------ work


def work(case):
    """State and springs read and written once, outputs written once, and the arithmetic of every step: 300 operations
    for a touching or bonded ordered pair, 45 for one that only attracts, 36 to integrate a particle."""
    if case["kind"] == "pool":
        n, close, far = case["systems"] * case["median"] * 1.6, 2.0, 1.9
    elif case["kind"] == "serve":
        span = case["n_high"] / case["n_low"]
        n, close, far = case["requests"] * (case["n_high"] - case["n_low"]) / math.log(span), 2.0, 1.9
    else:
        n = case["n"]
        close = 2.0 if case["shape"] == "aggregate" else 4.0
        far = n - 1.0 - close if case["pairs"] == "all" else (1.9 if case["shape"] == "aggregate" else 12.0)
    outputs = 96 if case["kind"] == "serve" else 144
    return {"bytes": n * (2 * 144 + 2 * 72 * close + outputs), "flops": n * case["steps"] * (300 * close + 45 * far + 36)}


# ----------------------------------------------------------------------- exact


def _dot(a, b):
    return (a[:, 0] * b[:, 0] + a[:, 1] * b[:, 1]) + a[:, 2] * b[:, 2]


def _cross(a, b):
    return np.stack([a[:, 1] * b[:, 2] - a[:, 2] * b[:, 1], a[:, 2] * b[:, 0] - a[:, 0] * b[:, 2],
                     a[:, 0] * b[:, 1] - a[:, 1] * b[:, 0]], axis=1)


def _unit(a):
    q = _dot(a, a)
    return a / np.where(q > 0.0, np.sqrt(q), 1.0)[:, None]


def _pairs_within(x, radius):
    """Ordered pairs (i, j), i != j, closer than radius (strictly), by i and then j."""
    n = len(x)
    c = np.floor((x - x.min(axis=0)) / (radius * (1.0 + 1e-9))).astype(np.int64) + 1
    span = c.max(axis=0) + 2
    key = (c[:, 0] * span[1] + c[:, 1]) * span[2] + c[:, 2]
    order = np.argsort(key, kind="stable")
    sorted_key = key[order]
    ii, jj = [], []
    for dx in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dz in (-1, 0, 1):
                other = key + (dx * span[1] + dy) * span[2] + dz
                lo, hi = np.searchsorted(sorted_key, other, "left"), np.searchsorted(sorted_key, other, "right")
                count = hi - lo
                i = np.repeat(np.arange(n), count)
                ii.append(i)
                jj.append(order[np.arange(count.sum()) - np.repeat(np.cumsum(count) - count, count) + np.repeat(lo, count)])
    i, j = np.concatenate(ii), np.concatenate(jj)
    d = x[i] - x[j]
    keep = (np.sqrt(_dot(d, d)) < radius) & (i != j)
    i, j = i[keep], j[keep]
    order = np.lexsort((j, i))
    return i[order], j[order]


def _forest(x, d_crit):
    """Bonds of touching pairs in row order, loop-closing ones left out: keys i * n + j of both directions."""
    n = len(x)
    i, j = _pairs_within(x, 2.0 * R + 2.0 * d_crit)
    d = x[i] - x[j]
    touch = (np.abs(np.sqrt(_dot(d, d)) - 2.0 * R) < d_crit) & (i < j)
    parent = list(range(n))

    def root(a):
        while parent[a] != a:
            parent[a] = parent[parent[a]]
            a = parent[a]
        return a

    keys = []
    for a, b in zip(i[touch].tolist(), j[touch].tolist()):
        ra, rb = root(a), root(b)
        if ra != rb:
            parent[rb] = ra
            keys += [a * n + b, b * n + a]
    return np.sort(np.array(keys, dtype=np.int64))


class _Springs:
    """Three spring vectors per ordered pair; a pair that is not held has zeros."""

    def __init__(self, keys=()):
        self.keys = np.array(keys, dtype=np.int64)
        self.s = np.zeros((3, len(self.keys), 3))

    def get(self, keys):
        out = np.zeros((3, len(keys), 3))
        if len(self.keys):
            at = np.minimum(np.searchsorted(self.keys, keys), len(self.keys) - 1)
            hit = self.keys[at] == keys
            out[:, hit] = self.s[:, at[hit]]
        return out

    def put(self, seen, keys, s):
        """New springs of the pairs `keys` out of the pairs `seen` this pass; the unseen keep theirs."""
        if len(self.keys):
            at = np.minimum(np.searchsorted(seen, self.keys), len(seen) - 1)
            old = seen[at] != self.keys
            keys, s = np.concatenate([keys, self.keys[old]]), np.concatenate([s, self.s[:, old]], axis=1)
        order = np.argsort(keys, kind="stable")
        self.keys, self.s = keys[order], s[:, order]


def _turn(xi, n):
    new = xi - _dot(xi, n)[:, None] * n
    length = np.sqrt(_dot(new, new))
    some = length > 0.0
    new[some] = new[some] / length[some][:, None] * np.sqrt(_dot(xi[some], xi[some]))[:, None]
    return new


def _slip_spring(xi, n, k, g, f_n, mu, phi, v, dt):
    xi = _turn(xi, n)
    f0 = (-k) * xi - g * v
    size = np.sqrt(_dot(f0, f0))
    t = f0 / np.where(size > 0.0, size, 1.0)[:, None]
    static, dynamic = mu * f_n, mu * phi * f_n
    stick = size <= static
    xi = np.where(stick[:, None], xi + v * dt, (-1.0 / k) * (dynamic[:, None] * t + g * v))
    limit = np.where(stick, static, dynamic)
    return np.where(size < limit, size, limit)[:, None] * t, xi


def _bond_spring(xi, n, k, g, v, dt):
    xi = _turn(xi, n)
    return (-k) * xi - g * v, xi + v * dt


def _hamaker_slope(A, h):
    return (-A) / 6.0 * ((((4.0 * R + 2.0 * h) / (4.0 * R + h) / h - 2.0 / (2.0 * R + h))
                          - 4.0 * (R * R) / ((2.0 * R + h) * (2.0 * R + h) * (2.0 * R + h)))
                         - 2.0 * (R * R) * (4.0 * R + 2.0 * h) / ((4.0 * R + h) * (4.0 * R + h)) / (h * h))


def _hamaker_energy(A, h):
    return (-A) / 6.0 * (2.0 * R * R / ((4.0 * R + h) * h) + 2.0 * R * R / (2.0 * R + h) ** 2
                         + np.log((4.0 * R + h) * h / (2.0 * R + h) ** 2))


class _Model:
    """The time stepping of one system: state, pair list, springs."""

    def __init__(self, case, seed):
        self.case, self.all = case, case["pairs"] == "all"
        self.x, self.v, self.w = _inputs(case, seed)
        self.n = len(self.x)
        self.theta = np.zeros_like(self.x)
        self.contact, self.bond, self.ham = _functors(case["binary"])
        sinter = case["binary"] == "sinter"
        self.bonds = _forest(self.x, self.bond[12]) if sinter else np.zeros(0, dtype=np.int64)
        self.springs = _Springs(self.bonds)
        if case["binary"] == "legacy":
            self.ends, self.arms = L.legacy_sinter_frames(self.x, R, 1.0e-9, _unit_vectors(seed))
            self.ends = self.ends.astype(np.int64)
        self.relist()
        self.a = None

    def relist(self):
        if self.all:
            i, j = np.divmod(np.arange(self.n * self.n), self.n)
            self.i, self.j = i[i != j], j[i != j]
        else:
            self.i, self.j = _pairs_within(self.x, self.case["r_list"] * R)

    def accelerate(self):
        i, j, x, v, w = self.i, self.j, self.x, self.v, self.w
        key = i * self.n + j
        d = x[i] - x[j]
        n = _unit(d)
        dist = _dot(d, n)
        bonded = np.isin(key, self.bonds)
        held = np.zeros(len(key), dtype=bool)
        if self.case["binary"] == "legacy":
            held = np.isin(key, np.concatenate([self.ends[:, 0] * self.n + self.ends[:, 1],
                                                self.ends[:, 1] * self.n + self.ends[:, 0]]))
        lin, ang = np.zeros((len(i), 3)), np.zeros((len(i), 3))
        springs = self.springs.get(key)
        keep = bonded.copy()
        for of, p in ((bonded, self.bond), (~bonded & ~held & (2.0 * R - dist > 0.0), self.contact)):
            at = np.flatnonzero(of)
            if not len(at):
                continue
            keep[at] = True
            ia, ja, m = i[at], j[at], n[at]
            k, g = (p[0], p[2], p[4], p[6]), (p[1], p[3], p[5], p[7])
            if p is self.contact:
                k, g = (p[0], p[2], p[6], p[10]), (p[1], p[3], p[7], p[11])
            overlap = 2.0 * R - dist[at]
            arm = R - overlap / 2.0
            f_n = k[0] * overlap + g[0] * -_dot(v[ia] - v[ja], m)
            ci, cj = _cross(m, w[ia]), _cross(m, w[ja])
            rel = ((v[ia] - v[ja]) + arm[:, None] * ci) + arm[:, None] * cj
            moves = (rel - _dot(rel, m)[:, None] * m, (-arm)[:, None] * (ci - cj),
                     (R * (_dot(m, w[ia]) - _dot(m, w[ja])))[:, None] * m)
            f = []
            for c in range(3):
                if p is self.contact:
                    got = _slip_spring(springs[c, at], m, k[c + 1], g[c + 1], f_n, p[4 + 4 * c], p[5 + 4 * c], moves[c], DT)
                else:
                    got = _bond_spring(springs[c, at], m, k[c + 1], g[c + 1], moves[c], DT)
                f.append(got[0])
                springs[c, at] = got[1]
            torque = (-(arm[:, None] * _cross(m, f[0])) + R * _cross(m, f[1])) + R * f[2]
            lin[at] = (f_n[:, None] * m + f[0]) / MASS
            ang[at] = torque / INERTIA
        if self.case["binary"] == "legacy":
            self.connectors(key, lin, ang)
        self.springs.put(key, key[keep], springs[:, keep])
        model = _hamaker(self.case)
        if model:
            r = -d
            h = np.maximum(np.sqrt(_dot(r, r)) - 2.0 * R, self.ham[1])
            pull = _hamaker_slope(self.ham[0], h)[:, None] * _unit(r) / MASS
            if model == "limited":
                pull[np.sqrt(_dot(d, d)) > self.ham[2]] = 0.0
            lin = lin + pull
        self.a, self.alpha = np.zeros_like(x), np.zeros_like(x)
        np.add.at(self.a, i, lin)
        np.add.at(self.alpha, i, ang)

    def connectors(self, key, lin, ang):
        """The five springs of each bond, seen from either end."""
        for one, two in ((0, 1), (1, 0)):
            a, b = self.ends[:, one], self.ends[:, two]
            at = np.searchsorted(key, a * self.n + b)
            force, torque = np.zeros((len(a), 3)), np.zeros((len(a), 3))
            for q in range(5):
                ca, cb = self.arms[:, one, q], self.arms[:, two, q]
                stretch = cb - ca
                length = np.sqrt(_dot(stretch, stretch))
                rest = 2.0 * R if q < 4 else 0.0
                rel = (self.v[b] + _cross(self.w[b], cb - self.x[b])) - (self.v[a] + _cross(self.w[a], ca - self.x[a]))
                f = (-(rest - length) * self.bond[0])[:, None] * _unit(stretch) + self.bond[1] * rel
                force, torque = force + f, torque + _cross(ca - self.x[a], f)
            lin[at], ang[at] = force / MASS, torque / INERTIA

    def step(self, steps, start):
        half, every = DT / 2.0, self.case.get("rebuild", 0)
        if self.a is None:
            self.accelerate()
        for s in range(start, start + steps):
            if every and not self.all and s % every == 0:
                self.relist()
            self.v, self.w = self.v + self.a * half, self.w + self.alpha * half
            self.x, self.theta = self.x + self.v * DT, self.theta + self.w * DT
            if self.case["binary"] == "legacy":
                for side in (0, 1):
                    own = self.ends[:, side]
                    for q in range(5):
                        p = self.arms[:, side, q] + self.v[own] * DT
                        self.arms[:, side, q] = p + _cross(self.w[own] * DT, p - self.x[own])
            self.accelerate()
            self.v, self.w = self.v + self.a * half, self.w + self.alpha * half

    def line(self):
        """Momenta and radius of gyration, then the energy ledger's terms and total."""
        x, v, w = self.x, self.v, self.w
        trans, rot = 0.5 * MASS * np.sum(v * v), 0.5 * INERTIA * np.sum(w * w)
        turn = np.sum(INERTIA * w + np.cross(x, MASS * v), axis=0)
        gyr = math.sqrt(np.sum((x - x.mean(axis=0)) ** 2) / self.n)
        d = x[self.i] - x[self.j]
        dist = np.sqrt(_dot(d, d))
        bonded = np.isin(self.i * self.n + self.j, self.bonds)
        overlap = 2.0 * R - dist
        normal = 0.25 * np.sum(np.where(bonded, self.bond[0] * overlap ** 2,
                                        np.where(overlap > 0.0, self.contact[0] * overlap ** 2, 0.0)))
        mine = np.isin(self.springs.keys, self.bonds)
        stored = [0.25 * np.sum(np.where(mine, self.bond[2 + 2 * c], self.contact[2 + 4 * c])
                                * _dot(self.springs.s[c], self.springs.s[c])) for c in range(3)]
        A, h0, cut = self.ham[:3]

        def potential(h):
            lower = _hamaker_energy(A, h0) + _hamaker_slope(A, h0) * (h - h0)
            return np.where(h < h0, lower, _hamaker_energy(A, np.maximum(h, h0)))

        pull = 0.5 * np.sum(np.where(dist > cut, 0.0, potential(dist - 2.0 * R) - potential(cut - 2.0 * R)))
        terms = [trans, rot, normal, *stored, pull]
        return [MASS * np.linalg.norm(v.sum(axis=0)), np.linalg.norm(turn), gyr, *terms, sum(terms)]


def exact(case, seed):
    """What run() returns, stepped in NumPy; None for facets and batches, which it does not model."""
    if case["kind"] in ("pool", "serve") or case.get("plates"):
        return None
    if case["n"] * case["steps"] > (60 if case["pairs"] == "all" else 100) * 20000:
        return None
    m = _Model(case, seed)
    every = case.get("every", case["steps"])
    lines = []
    for s in range(0, case["steps"], every):
        m.step(min(every, case["steps"] - s), s)
        if case["kind"] == "ledger":
            lines.append(m.line())
    out = dict(x=m.x, v=m.v, theta=m.theta, omega=m.w, a=m.a, alpha=m.alpha)
    return dict(out, **_columns(lines)) if lines else out
