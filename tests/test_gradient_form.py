"""The bracket D of dW/dq in the FP64 gradient sweep and force pass, evaluated on the host from the
library's own header, against exact arithmetic: dW/dq vanishes with q, so D has to be exact relative to
itself down to the smallest q (the truncated powers 81 - 96 + 15 of the quintic kernel leave 1e-9 at
q = 1e-6), as the reference's inner piece is.

Tolerances, u = 2^-53: quintic, below 1: four roundings of a polynomial between 10 and 24 that its terms
do not exceed 58, 4 * 58 / 10 u; above: a^4 with 2-u roundings each of a (four times), a^2 and a^4, over
a^4 - 6 b^4 >= 10/16 of it: 16 u; taken as 24 u.  Cubic, whose inner piece the reference has as
truncated powers, 4 - 4 at q = 0: relative to 1, eight roundings of terms of at most 2."""
import os
import shutil
import subprocess
from fractions import Fraction as F

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
U = 2.0 ** -53


def _exact(q, kernel):
    q = F(q)
    up = lambda c: max(c - q, F(0))  # noqa: E731
    if kernel == "quintic":
        return up(3) ** 4 - 6 * up(2) ** 4 + 15 * up(1) ** 4
    return up(2) ** 2 - 4 * up(1) ** 2


@pytest.mark.parametrize("kernel,radius", [("cubic", 2.0), ("quintic", 3.0)])
def test_gradient_bracket(kernel, radius, tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    exe = str(tmp_path / "gf")
    flags = ["-DCOSMO_KERNEL_QUINTIC"] if kernel == "quintic" else []
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O2", "-std=c++17", *flags,
                    os.path.join(HERE, "native", "gradient_form.cpp"), "-o", exe], check=True, capture_output=True)
    rng = np.random.default_rng(3)
    q = np.concatenate([10.0 ** rng.uniform(-12, 0, 2000), rng.uniform(0, radius, 4000), np.nextafter([1.0, 2.0], 0.0),
                        [0.0, 1.0, 2.0, radius]])
    text = "\n".join("%.17g" % v for v in q)
    out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout
    got = np.array([line.split() for line in out.strip().split("\n")], dtype=float)
    for v, (d, d2) in zip(q, got):
        assert d == d2
        e = _exact(v, kernel)
        if kernel == "quintic":
            assert abs(F(d) - e) <= F(24 * U) * e, (v, d)
        else:
            assert abs(F(d) - e) <= F(16 * U), (v, d)
