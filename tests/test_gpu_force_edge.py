"""Pairs at the edge of a support, q = R up to rounding, in the FP64 force pass: the sound speed of such a
pair enters the maximum of the signal speed or does not, so the test has to round as the reference's
does (r^2 / h^2 < R^2, not r / h < R).  Simple cubic lattices whose second neighbours lie at R h to a few
units in the last place; signal speeds against the oracle's at the same h, where one pair more or less shows
as a difference of order one."""
import numpy as np
import pytest

from cosmosphere_amd import Library, workloads
from cosmosphere_amd.api import FORCE_OUT, HSML, THERMO
from gpu_common import DEFAULT_ITEMS
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spacing", [0.6966794926011195, 0.893185797606609, 0.11080095245394586])
def test_edge_of_support(spacing):
    rng = np.random.default_rng(5)
    g = np.arange(9) * spacing
    x = np.stack(np.meshgrid(g, g, g, indexing="ij")).reshape(3, -1)
    n = x.shape[1]
    c = workloads._pack(*x, np.full(n, 1.2 * spacing), "cubic", "lattice")
    h = spacing * (1.0 + rng.integers(-3, 4, n) * 2.0 ** -52)        # R h = 2 spacings
    v = rng.standard_normal((3, n))
    th = np.stack([np.ones(n), rng.uniform(1.0, 2.0, n), np.ones(n), np.ones(n)])
    print("case edge", spacing, flush=True)
    lib = Library("cubic")
    for k, val in DEFAULT_ITEMS.items():
        lib.set_option(k, val)
    lib.set_option("precision", 0)
    lib.solve(c["x"], c["y"], c["z"], c["h"], spacing ** 3, hfact=1.2, v=v)
    lib.upload(HSML, h)
    lib.upload_sorted(THERMO, th)
    lib.force(n, spacing ** 3, beta=2.0, alphau=1.0)
    vsig = lib.download(FORCE_OUT, n)[4]
    o = O.Oracle(quintic=False)
    o.set_particles(c["x"], c["y"], c["z"], c["h"], v=v, a=np.zeros((3, n)))
    o.build()
    order = o.get("order")
    o.set_h_sorted(h[order])
    o.set_gradh_sorted(np.zeros(n))
    o.hmax_all()
    o.build_lists(symmetric=True)
    o.set_thermo(*th)
    o.force(spacing ** 3, 1.2, beta=2.0, alphau=1.0)
    ref = np.empty(n)
    ref[order] = o.get("vsig")
    np.testing.assert_allclose(vsig, ref, rtol=1e-12, atol=0.0)
