"""The force pass's culling of list entries (keep, force.hip), which runs for every lane of a wavefront
and reads the chunk's particles from other lanes: lists shorter than a wavefront, a little longer, and of
several rounds with a partial last one, leaves from one particle to more than 64.  Against the oracle
on the same tree, in the tolerances of test_gpu_force.py."""
import numpy as np
import pytest

from cosmosphere_amd import Library, workloads
from cosmosphere_amd.api import FORCE_OUT, THERMO
from gpu_common import DEFAULT_ITEMS
from oracle import oracle as O
from test_gpu_force import thermo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("bucket", [8, 32, 128])
@pytest.mark.parametrize("npartx", [4, 7, 14])
def test_list_lengths(npartx, bucket, precision):
    c = workloads.config2(npartx=npartx)
    n = c["n"]
    rng = np.random.default_rng(npartx)
    v, u = 0.1 * rng.standard_normal((3, n)), 1.0 + 0.5 * rng.random(n)
    print("case lists", npartx, bucket, precision, flush=True)
    lib = Library(c["kernel"])
    for k, val in DEFAULT_ITEMS.items():
        lib.set_option(k, val)
    lib.set_option("bucket", bucket)
    lib.set_option("precision", precision)
    try:
        out = lib.solve(c["x"], c["y"], c["z"], c["h"], c["pmass"], hfact=c["hfact"], v=v)
        th = thermo(c, out["h"], u)
        lib.upload_sorted(THERMO, th)
        lib.force(n, c["pmass"], beta=2.0, alphau=1.0)
        f = lib.download(FORCE_OUT, n)
    finally:
        lib.set_option("bucket", 64)
        lib.set_option("precision", 0)
    o = O.Oracle(quintic=False, bucket=bucket)
    o.set_particles(c["x"], c["y"], c["z"], c["h"], v=v, a=np.zeros((3, n)))
    o.build()
    assert o.density_solve(c["pmass"], 1e-4, c["hfact"], 100, 0, True) == 0
    o.set_thermo(*th)
    o.force(c["pmass"], c["hfact"], beta=2.0, alphau=1.0)
    order = o.get("order")
    tol = 1e-9 if precision == 0 else 2e-6
    for rows, names in (((0, 1, 2), ("fx", "fy", "fz")), ((3,), ("du",)), ((5,), ("divvF",))):
        ref = np.empty((len(rows), n))
        ref[:, order] = np.stack([o.get(m) for m in names])
        assert np.max(np.abs(f[list(rows)] - ref)) < tol * np.abs(ref).max(), names
