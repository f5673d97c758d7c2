"""The total of a pass's neighbour-leaf lists against the list buffer's capacity, around 2^32
entries: the 32-bit offsets wrap there, and a total that wrapped with them would pass for one that fits, so
that the fill would write far past the buffer.  tests/native/list_scan.cpp runs the scans alone."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXE = os.path.join(ROOT, "cosmosphere_amd", "lib", "list_scan_check")


@pytest.mark.gpu
def test_totals_beyond_32_bits():
    res = subprocess.run([EXE], capture_output=True, text=True, timeout=100)
    assert res.returncode == 0, res.stdout + res.stderr
    assert res.stdout.count("entries") == 16 and "WRONG" not in res.stdout
