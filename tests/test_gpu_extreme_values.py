"""Positions and radii at the ends of the number range: the kernels' squared
distance tests must not decide what the functors decide with a distance."""
import numpy as np
import pytest

import _oracle as O

pytestmark = pytest.mark.gpu

R = O.R_PART


@pytest.mark.parametrize("pairs", [0, 1])
@pytest.mark.parametrize("far", [np.inf, -np.inf, np.nan, 1e160])
@pytest.mark.parametrize("n", [6, 40])
def test_a_lost_particle_acts_as_the_contact_functor_says(n, far, pairs):
    """A particle at infinity has no direction and overlaps everything it is
    paired with by a NaN; one whose squared distance overflows, by a diameter.
    Tiny systems and tiles, all pairs and a list made while it was near."""
    import libgran_amd as L
    print(f"[extreme] n {n}, far {far}, pairs {pairs}", flush=True)
    g = np.arange(n)
    x = np.stack([g % 4, g // 4 % 4, g // 16], axis=1) * 2.0 * R
    kw = dict(r_verlet=3.2 * R) if pairs else {}
    o = O.OracleSystem(O.system_params(O.BIN_CONTACT, O.HAM_NONE, neighbor_mode=pairs, contact=O.contact_params(), **kw), x)
    s = L.System(L.make_params(L.BINARY_CONTACT, L.HAMAKER_NONE, pair_mode=pairs, contact=O.contact_params(),
                               pair_capacity=n, **kw), x)
    y = x.copy()
    y[3, 0] = far
    o.set_state(x=y)
    s.set_state(x=y)
    o.compute_accelerations()
    s.compute_accelerations()
    a, b = o.state(), s.state()
    for k in ("a", "alpha"):
        np.testing.assert_array_equal(b[k], a[k], err_msg=k)
    np.testing.assert_array_equal(s.springs(0)[0], o.springs(0)[0])
    o.step(1e-13, 1)
    if np.all(np.isfinite(o.state()["v"])):
        s.step(1e-13, 1)
        np.testing.assert_array_equal(s.state()["v"], o.state()["v"])
    else:
        with pytest.raises(L.HipgranError) as e:
            s.step(1e-13, 1)
        assert e.value.status == 4  # HG_ERR_NUMERIC
    s.close()


@pytest.mark.parametrize("n", [32, 300])
def test_radii_whose_squares_underflow(n):
    """Overlaps and list radii of 1e-161: their squares have a few bits left."""
    import libgran_amd as L
    print(f"[extreme] small radii, n {n}", flush=True)
    tiny = 1e-161
    rng = np.random.default_rng(n)
    x = rng.uniform(0.0, 2.5 * tiny, (n, 3))
    contact = O.contact_params(gamma_n=0.0, dt=1e-3, r_part=0.5 * tiny, mass=1.0, inertia=1.0)
    for pairs in (0, 1):
        kw = dict(r_verlet=2.0 * tiny, neighbor_capacity=n) if pairs else {}
        o = O.OracleSystem(O.system_params(O.BIN_CONTACT, O.HAM_NONE, neighbor_mode=pairs, contact=contact,
                                           **({k: v for k, v in kw.items() if k == "r_verlet"})), x)
        s = L.System(L.make_params(L.BINARY_CONTACT, L.HAMAKER_NONE, pair_mode=pairs, contact=contact, pair_capacity=n,
                                   **kw), x)
        if pairs:
            o.rebuild()
            np.testing.assert_array_equal(s.neighbors()[0], o.neighbors()[0])
            np.testing.assert_array_equal(s.neighbors()[1], o.neighbors()[1])
        o.step(1e-3, 2)
        s.step(1e-3, 2)
        np.testing.assert_array_equal(s.springs(0)[0], o.springs(0)[0])
        np.testing.assert_array_equal(s.state()["a"], o.state()["a"])
        s.close()
