"""Device bytes that a pool is said to take per particle."""
import _oracle as O


def test_all_pairs_pools_count_their_block_map():
    """At least, with all pairs: nine fields of four doubles, both halves of a table of 24
    entries (tag and ten doubles) and counts, the owner, and a 16-byte block of
    the per-step launches for every particle."""
    import libgran_amd as L
    none = L.make_params(L.BINARY_NONE, L.HAMAKER_FULL, hamaker=O.hamaker_params())
    contact = L.make_params(L.BINARY_CONTACT, L.HAMAKER_FULL, contact=O.contact_params(), hamaker=O.hamaker_params())
    assert L.Pool.bytes_per_particle(none, 0) >= 9 * 32 + 2 * 4 + 4 + 16
    assert L.Pool.bytes_per_particle(contact, 0) >= 9 * 32 + 2 * (24 * 84 + 4) + 4 + 16
