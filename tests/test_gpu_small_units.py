"""The FP64 gradient sweep in code units so small that separations come near the reference's guard eps =
2.2e-16 of 1 / (r + eps), down to separations below it, against the oracle.  Scaling positions and h
by a power of two leaves every other digit of the sums as it is, so the tolerance is that of the parity
test of the sweep at the ordinary scale.  A tenth of the particles sit at q of about 1e-6 from another one."""
import numpy as np
import pytest

from cosmosphere_amd import Library, workloads
from gpu_common import DEFAULT_ITEMS, oracle_run, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel", ["cubic", "quintic"])
@pytest.mark.parametrize("power", [0, -27, -34, -44, -52])
def test_small_units(kernel, power):
    rng = np.random.default_rng(17)
    n, hfact = 3000, 1.2 if kernel == "cubic" else 1.0
    x = rng.random((3, n))
    h = np.full(n, hfact * n ** (-1.0 / 3.0))
    k = n // 10
    x[:, :k] = x[:, k:2 * k] + 1e-6 * h[0] * rng.standard_normal((3, k))
    scale = 2.0 ** power
    c = workloads._pack(x[0] * scale, x[1] * scale, x[2] * scale, h * scale, kernel, "uniform")
    v = np.stack([0.3 * x[0] - 0.1 * x[1], 0.2 * x[2] + 0.05 * x[0], -0.4 * x[1]])
    a = np.stack([np.sin(3 * x[0]), np.cos(2 * x[1]), x[2] ** 2])
    print("case units", kernel, power, flush=True)
    lib = Library(kernel)
    for key, val in DEFAULT_ITEMS.items():
        lib.set_option(key, val)
    lib.set_option("precision", 0)
    out = lib.solve(c["x"], c["y"], c["z"], c["h"], c["pmass"], tolh=1e-4, hfact=c["hfact"], v=v, a=a)
    o, unconv = oracle_run(c, v=v, a=a)
    assert unconv == 0
    order = o.get("order")
    for f in ("h", "rho", "divv", "ddivvdt"):
        ref = np.empty(n)
        ref[order] = o.get(f)
        assert rel_err(out[f], ref, floor=np.abs(ref).max() * 1e-6) < 1e-7, f
