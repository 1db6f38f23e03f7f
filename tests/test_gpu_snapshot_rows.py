"""Legacy connector rows of a snapshot that differ from its bond list: the rows
are what a step reads, so they, and not the bonds, say how much the
tiny-system kernel keeps in LDS; slots beyond the table are refused."""
import struct

import numpy as np
import pytest

import _oracle as O
import _scenarios as S

pytestmark = pytest.mark.gpu

R = O.R_PART


def sealed(body):
    """Snapshot bytes with their FNV-1a hash."""
    h = 1469598103934665603
    for b in body:
        h = (h ^ b) * 1099511628211 % (1 << 64)
    return bytes(body) + struct.pack("<Q", h)


class Layout:
    """Offsets in a legacy system's snapshot without a neighbour list (snapshot.h)."""

    def __init__(self, raw):
        self.counts = 16 + struct.unpack_from("<I", raw, 12)[0] + 24 + 32
        n, = struct.unpack_from("<Q", raw, self.counts - 56)
        self.nbonds, _, _, pt, _, self.legacy = struct.unpack_from("<6Q", raw, self.counts)
        self.bonds = self.counts + 48 + 6 * 24 * n + 4 * n + 76 * pt
        self.leg_slot = self.bonds + 8 * self.nbonds + 4 * n + 4 * self.legacy
        assert self.leg_slot + 124 * self.legacy + 8 == len(raw)


def lattice():
    import libgran_amd as L
    x, v = S.sinter_lattice()
    s13 = O.sinter_params(k_bond=1.0e4, d_crit=1.0e-9)
    s13[1] = 0.0
    s = L.System(L.make_params(L.BINARY_SINTER_LEGACY, L.HAMAKER_NONE, contact=O.contact_params(), sinter=s13), x, v)
    vecs = np.random.default_rng(5).uniform(-1.0, 1.0, (5000, 3))
    pairs, conn, _ = O.legacy_frames(x, R, 1.0e-9, vecs / np.linalg.norm(vecs, axis=1)[:, None])
    s.set_legacy_connectors(pairs, conn)
    return s


def test_rows_without_bonds_step_as_they_are():
    import libgran_amd as L
    print("[snapshot] legacy rows without bonds", flush=True)
    s = lattice()
    raw = s.save()
    y = Layout(raw)
    body = bytearray(raw[:y.bonds] + raw[y.bonds + 8 * y.nbonds:-8])
    struct.pack_into("<Q", body, y.counts, 0)
    t = L.System.load(sealed(body))
    s.step(1e-13, 500)
    t.step(1e-13, 500)
    a, b = s.state(), t.state()
    for k in ("x", "v", "theta", "omega", "a", "alpha"):
        np.testing.assert_array_equal(b[k], a[k], err_msg=k)


@pytest.mark.parametrize("slot", [16, 1 << 20, 0xffffffff])
def test_slots_beyond_the_table_are_refused(slot):
    import libgran_amd as L
    print(f"[snapshot] legacy slot {slot}", flush=True)
    raw = lattice().save()
    body = bytearray(raw[:-8])
    struct.pack_into("<I", body, Layout(raw).leg_slot + 4, slot)
    with pytest.raises(L.HipgranError, match="bad legacy rows"):
        L.System.load(sealed(body))
