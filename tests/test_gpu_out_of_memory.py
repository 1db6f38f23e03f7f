"""A system whose second set of buffers does not fit says so and steps on once
there is room: each of the allocations of its first step is refused in turn, in
a program whose hipMalloc counts (tests/cpp/malloc_limit.cpp)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))

PROGRAM = """
import ctypes, sys
limit = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL).malloc_limit
import numpy as np
import libgran_amd as L, _oracle as O, _scenarios as S
x = L.generate_aggregate(70, O.R_PART, 1.8, 1.3, 3)
v = np.random.default_rng(3).normal(0.0, 1.0, x.shape)
c, sn, h = S.aggregate_params()
p = L.make_params(L.BINARY_SINTER, L.HAMAKER_LIMITED, pair_mode=1, r_verlet=3.2 * O.R_PART, contact=c, sinter=sn, hamaker=h)
states = []
refused = 0
for call in (-1, 0, 1, 2, 3, 4, 5):
    s = L.System(p, x, v)
    limit(call)
    try:
        s.step(1e-13, 7, rebuild_every=5)
    except L.HipgranError as e:
        assert e.status == 2, e  # HG_ERR_OOM
        refused += 1
        limit(-1)
        s.step(1e-13, 7, rebuild_every=5)
    limit(-1)
    states.append(s.state())
    s.close()
for k in states[0]:
    for t in states[1:]:
        np.testing.assert_array_equal(t[k], states[0][k], err_msg=k)
assert refused >= 3, refused
print("refused", refused)
"""


def test_a_refused_first_step_is_taken_later():
    print("[oom] first step", flush=True)
    subprocess.run(["make", "-s", "-C", os.path.join(HERE, "cpp"), "build/libmalloc_limit.so"], check=True)
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([os.path.dirname(HERE), HERE]))
    r = subprocess.run([sys.executable, "-c", PROGRAM, os.path.join(HERE, "cpp", "build", "libmalloc_limit.so")],
                       capture_output=True, text=True, env=env, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "refused" in r.stdout
