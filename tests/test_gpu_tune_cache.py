"""The autotuner's file (COSMO_TUNE_CACHE): a choice is taken again by another process, and a line that a
build with other kernels wrote (a signature without their number, where loop_blocks_scale scaled another
grid) is not."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import sys
import numpy as np
sys.path[:0] = [%r, %r]
from cosmosphere_amd import Library
from cosmosphere_amd.api import HSML, POS
from gpu_common import dataset
c = dataset("tiny")
lib = Library(c["kernel"])
n = c["n"]
lib.arrays_init(n)
lib.upload(POS, np.stack([c["x"], c["y"], c["z"]]))
lib.upload(HSML, c["h"])
got = lib.autotune(n, c["pmass"], tolh=1e-4, hfact=c["hfact"], budget_s=0.2)
print("cached", int(got["tune_cached"]), "scale", int(got["loop_blocks_scale"]))
""" % (ROOT, os.path.join(ROOT, "tests"))


def _tune(path):
    res = subprocess.run([sys.executable, "-c", CHILD], capture_output=True, text=True, timeout=100,
                         env=dict(os.environ, COSMO_TUNE_CACHE=path))
    assert res.returncode == 0, res.stdout + res.stderr
    return next(ln.split() for ln in res.stdout.splitlines() if ln.startswith("cached"))


def test_file_of_another_build(tmp_path):
    path = str(tmp_path / "tune")
    print("case tune: first process", flush=True)
    assert _tune(path)[1] == "0"
    sig, options = open(path).read().rstrip("\n").split("\t")
    print("case tune: same build again", flush=True)
    again = _tune(path)
    assert again[1] == "1" and "loop_blocks_scale=" + again[3] in options
    old = sig.rsplit(" kernels=", 1)[0]
    with open(path, "w") as f:
        f.write(old + "\t" + options + "\n")
    print("case tune: another build's line", flush=True)
    assert _tune(path)[1] == "0"
    assert open(path).read().startswith(old + "\t")
