"""The legacy sinter_functor over the range of its kernels: blocks of 27 (the
tiny-system kernel), 64 and 216 (one particle a thread) and 343 spheres (a launch
per step), in calls of odd and even lengths, against the oracle bit for bit."""
import numpy as np
import pytest

import _oracle as O

pytestmark = pytest.mark.gpu

R = O.R_PART


@pytest.mark.parametrize("pairs", [0, 1])
@pytest.mark.parametrize("m", [3, 4, 6, 7])
def test_blocks_equal_the_oracle(m, pairs):
    import libgran_amd as L
    print(f"[legacy] block of {m ** 3}, pairs {pairs}", flush=True)
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), axis=-1).reshape(-1, 3)
    x = np.concatenate([g[:-1] * 2.0 * R, [[m * 2.0 * R + 1.2e-9, 0.0, 0.0]]])  # the last one apart
    v = np.random.default_rng(m).normal(0.0, 0.5, x.shape)
    v[-1] = [-100.0, 0.0, 0.0]
    s13 = O.sinter_params(k_bond=1.0e4, d_crit=1.0e-9)
    s13[1] = 0.0
    vecs = np.random.default_rng(5).uniform(-1.0, 1.0, (200 * m ** 3, 3))
    conn = O.legacy_frames(x, R, 1.0e-9, vecs / np.linalg.norm(vecs, axis=1)[:, None])[:2]
    kw = dict(r_verlet=4.0 * R) if pairs else {}
    o = O.OracleSystem(O.system_params(O.BIN_SINTER_LEGACY, O.HAM_NONE, neighbor_mode=pairs, contact=O.contact_params(),
                                       sinter=s13, **kw), x, v)
    o.set_legacy(*conn)
    s = L.System(L.make_params(L.BINARY_SINTER_LEGACY, L.HAMAKER_NONE, pair_mode=pairs, contact=O.contact_params(),
                               sinter=s13, **kw), x, v)
    s.set_legacy_connectors(*conn)
    held = 0
    for steps in (1, 2, 37, 45, 55, 40):
        o.step(1e-13, steps, rebuild_every=20 * pairs)
        s.step(1e-13, steps, rebuild_every=20 * pairs)
        a, b = o.state(), s.state()
        for k in ("x", "v", "theta", "omega", "a", "alpha"):
            np.testing.assert_array_equal(b[k], a[k], err_msg=f"{k} after {steps}")
        np.testing.assert_array_equal(s.springs(0)[0], o.springs(0)[0])
        np.testing.assert_array_equal(s.springs(0)[1], o.springs(0)[1])
        held = max(held, len(o.springs(0)[0]))
    assert held > 0  # the last sphere touched the block
    s.close()
