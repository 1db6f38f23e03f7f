"""The one-workgroup kernel of tiny systems against the CPU oracle at the
sizes of its range, with contacts that begin and end, lists that leave table
entries out, and interval lengths of one step and more. FP64: equal to the last
bit."""
import numpy as np
import pytest

import _oracle as O
from test_gpu_tile_step import hot_cloud

pytestmark = pytest.mark.gpu

R = O.R_PART


@pytest.mark.parametrize("pairs,r_list", [("all", 0.0), ("list", 5.0), ("list", 2.02)])
@pytest.mark.parametrize("n", [1, 2, 3, 8, 17, 31, 32, 33])
def test_tiny_equals_oracle(n, pairs, r_list):
    """33 particles are past the kernel's range. A list of 2.02 r loses and
    regains touching partners between rebuilds, whose springs are carried."""
    import libgran_amd as L
    print(f"[tiny] n {n}, pairs {pairs} {r_list}", flush=True)
    x, v, w = hot_cloud(n, 100 + n)
    mode = 1 if pairs == "list" else 0
    kw = dict(r_verlet=r_list * R) if mode else {}
    ham = O.hamaker_params(A=1e-20, h0=1e-9)
    o = O.OracleSystem(O.system_params(O.BIN_CONTACT, O.HAM_FULL, neighbor_mode=mode, contact=O.contact_params(),
                                       hamaker=ham, **kw), x, v, w0=w)
    s = L.System(L.make_params(L.BINARY_CONTACT, L.HAMAKER_FULL, pair_mode=mode, contact=O.contact_params(),
                               hamaker=ham, **kw), x, v, omega0=w)
    every = 20 if mode else 0
    for steps in (1, 1, 2, 96, 60):
        o.step(1e-13, steps, rebuild_every=every)
        s.step(1e-13, steps, rebuild_every=every)
        a, b = o.state(), s.state()
        for k in ("x", "v", "theta", "omega", "a", "alpha"):
            np.testing.assert_array_equal(b[k], a[k], err_msg=f"{k} after {steps}")
        (ij1, s1), (ij2, s2) = o.springs(0), s.springs(0)
        np.testing.assert_array_equal(ij2, ij1)
        np.testing.assert_array_equal(s2, s1)
    s.close()


@pytest.mark.parametrize("pairs", ["all", "list"])
@pytest.mark.parametrize("per_step", [False, True])
def test_a_row_that_overflows_for_a_while_is_reported(per_step, pairs):
    """Two spheres bounce off a third from both sides within one call: for some
    steps its row needs two entries, at the end of the call none."""
    import libgran_amd as L
    print(f"[tiny] passing overflow, per step {per_step}, {pairs}", flush=True)
    gap = 2.0 * R + 2e-11
    x = np.array([[0.0, 0.0, 0.0], [gap, 0.0, 0.0], [-gap, 0.0, 0.0]])
    v = np.array([[0.0, 0.0, 0.0], [-10.0, 0.0, 0.0], [10.0, 0.0, 0.0]])
    mode = 1 if pairs == "list" else 0
    kw = dict(r_verlet=3.0 * R) if mode else {}
    o = O.OracleSystem(O.system_params(O.BIN_CONTACT, O.HAM_NONE, neighbor_mode=mode, contact=O.contact_params(), **kw), x, v)
    most = 0
    for _ in range(200):
        o.step(1e-13, 1)
        most = max(most, int(np.bincount(o.springs(0)[0][:, 0], minlength=3)[0]))
    assert most == 2 and len(o.springs(0)[0]) == 0
    for capacity in (1, 2):
        s = L.System(L.make_params(L.BINARY_CONTACT, L.HAMAKER_NONE, pair_mode=mode, contact=O.contact_params(),
                                   pair_capacity=capacity, **kw), x, v)
        s.per_step_launches(per_step)
        if capacity == 1:
            with pytest.raises(L.HipgranError, match="needs 2 slots per particle, capacity is 1") as e:
                s.step(1e-13, 200)
            assert e.value.status == 5  # HG_ERR_CAPACITY
        else:
            s.step(1e-13, 200)
            np.testing.assert_array_equal(s.state()["x"], o.state()["x"])
        s.close()
