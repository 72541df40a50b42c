"""The copies of results to the host (csrc/readback.hpp), with a runtime whose
streams end when the test says so."""
import os
import subprocess

import pytest

HOST = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host")


@pytest.fixture(scope="module")
def readback(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("readback") / "readback_host")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-Wno-attributes", "-I", HOST,
                    os.path.join(HOST, "readback_host.cpp"), "-o", exe], check=True)
    return exe


def check(exe, case):
    got = subprocess.run([exe, case], capture_output=True, text=True, timeout=100)
    assert got.returncode == 0, got.stdout


def test_copies_of_different_streams_overlap(readback):
    """A copy does not wait for the stream of another one, small or in chunks."""
    check(readback, "overlap")


def test_page_locked_memory_is_bounded_and_given_back(readback):
    """24 threads copy at once, sizes at and around a slot and beyond a set."""
    check(readback, "many")


def test_the_failure_of_a_copy_is_reported(readback):
    """What a launch or the stream failed with reaches the caller, from every thread of a copy."""
    check(readback, "errors")


def test_copies_with_another_device_current(readback):
    """The stream's device need not be the one that is current in the thread that reads."""
    check(readback, "devices")
