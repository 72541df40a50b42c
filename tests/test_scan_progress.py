"""The device-wide scan waits between blocks; here its code runs on the host (a
block's threads as fibers), one block after the other in any order of dispatch."""
import os
import subprocess

import pytest

HOST = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host")


@pytest.fixture(scope="module")
def scan(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("scan") / "scan_progress")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wno-attributes", "-I", HOST, os.path.join(HOST, "scan_progress.cpp"), "-o", exe],
                   check=True)
    return exe


@pytest.mark.parametrize("order", ["0", "1", "12345"])
@pytest.mark.parametrize("rows,n", [(4, 1), (4, 4096), (4, 4097), (4, 24581), (8, 8193), (8, 40961), (16, 16385),
                                    (16, 65537), (4, 258 * 4096 + 3)])
def test_every_wait_of_the_scan_ends(scan, rows, n, order):
    """A block waits only for blocks that began before it, whatever the order in
    which a launch's blocks begin and however few of them fit the chip, and the
    sums are right: one tile, a tile and one item, several tiles of each size, and
    more than a look-back's 256."""
    got = subprocess.run([scan, str(rows), str(n), order], capture_output=True, text=True, timeout=100)
    assert got.returncode == 0, got.stdout
