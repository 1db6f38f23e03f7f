"""Lookups in the tiles' pair-state rows (libgran_amd/csrc/pair_row.h), on the
host."""
import os
import subprocess

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")


def run(name):
    subprocess.run(["make", "-s", "-C", HERE, f"build/{name}"], check=True)
    p = subprocess.run([os.path.join(HERE, "build", name)], capture_output=True, text=True)
    assert p.returncode == 0, p.stdout


def test_an_entry_is_found_in_its_own_slot():
    """An entry that stays is found in its slot while other threads claim the
    slots behind the row, where its old tag may still stand; slots of rows
    longer than 4,095 entries keep their number in a tile's queue."""
    run("pair_row_check")
