"""Neighbour lists against the CPU oracle where their builders change: the
brute-force builder's tile and wavefront edges, the cell builder above its
line, lists longer than its LDS row, and a system far from the origin."""
import numpy as np
import pytest

import _oracle as O

pytestmark = pytest.mark.gpu

R = O.R_PART


def check(x, r_list, capacity=0):
    import libgran_amd as L
    print(f"[lists] n {len(x)}, r_list {r_list / R:.2f} r", flush=True)
    ham = O.hamaker_params()
    o = O.OracleSystem(O.system_params(O.BIN_NONE, O.HAM_LIMITED, neighbor_mode=1, r_verlet=r_list, hamaker=ham), x,
                       np.zeros_like(x))
    s = L.System(L.make_params(L.BINARY_NONE, L.HAMAKER_LIMITED, pair_mode=1, r_verlet=r_list, hamaker=ham,
                               neighbor_capacity=capacity), x)
    (off1, idx1), (off2, idx2) = o.neighbors(), s.neighbors()
    np.testing.assert_array_equal(off2, off1)
    np.testing.assert_array_equal(idx2, idx1)
    s.close()
    return off1


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 64, 65, 255, 256, 257, 513, 2047, 2048, 2049, 9001])
def test_lists_equal_oracle(n):
    rng = np.random.default_rng(n)
    side = 2.2 * R * n ** (1.0 / 3.0)
    check(rng.uniform(0.0, side, (n, 3)) - 0.5 * side, 3.2 * R)


@pytest.mark.parametrize("shift", [0.0, 1.0])
def test_cell_lists_longer_than_their_lds_row(shift):
    """About 200 partners each, and the same cloud a metre from the origin."""
    n = 9000
    rng = np.random.default_rng(5)
    x = rng.uniform(0.0, 2.0 * R * n ** (1.0 / 3.0), (n, 3)) + shift
    off = check(x, 7.0 * R, capacity=600)
    assert np.diff(off).max() > 96


def test_cell_lists_far_from_the_origin():
    n = 9000
    x = np.random.default_rng(6).uniform(0.0, 2.2 * R * n ** (1.0 / 3.0), (n, 3)) + np.array([1.0, -3.0, 0.1])
    check(x, 3.2 * R)


@pytest.mark.parametrize("where", [1.0, -1.0, np.inf])
def test_one_particle_far_away_leaves_the_others_listed(where):
    """A first particle 1e8 m out (or lost) beside pairs just inside the list
    radius: the cells of the others must not depend on it."""
    rng = np.random.default_rng(8)
    m, r_list = 1500, 3.2 * R
    a = rng.uniform(0.0, 40.0 * r_list, (m, 3))
    b = a.copy()
    b[np.arange(m), rng.integers(0, 3, m)] += r_list * (1.0 - 1e-5)
    out = where * np.array([[1e8, 0.7e8, -0.3e8]])
    off = check(np.concatenate([out, a, b]), r_list)
    assert off[-1] >= 2 * m
