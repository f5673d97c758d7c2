"""What the FP64 density pairs are made of, evaluated on the host from the library's own header: their
sums may be no less exact than those of the reference's pieces with the library's root, and their root
has to be the nearest double.

Tolerances: over 20,000 sets an rms error is known to 1/sqrt(40,000) = 0.5%, a ratio of two to 0.7%;
taken as 2%.  The root's last operation adds a correction of at most 2^-23 of it that is wrong by some
2^-52 of itself: it rounds the wrong way once in 2^22; taken as once in 10^4."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("kernel", ["cubic", "quintic"])
def test_sums_and_root(kernel, tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    exe = str(tmp_path / "df")
    flags = ["-DCOSMO_KERNEL_QUINTIC"] if kernel == "quintic" else []
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O2", "-mfma", "-std=c++17", *flags,
                    os.path.join(HERE, "native", "density_forms.cpp"), "-o", exe], check=True, capture_output=True)
    lines = [ln.split() for ln in subprocess.run([exe], capture_output=True, text=True, check=True).stdout.splitlines()]
    sums = [[float(v) for v in ln[1:]] for ln in lines if ln[0] == "sums"]
    assert len(sums) == 3
    for n, w0, w1, g0, g1 in sums:
        assert w1 <= 1.02 * w0, (n, w0, w1)
        assert g1 <= 1.02 * g0, (n, g0, g1)
    _, samples, wrong = next(ln for ln in lines if ln[0] == "root")
    assert int(wrong) <= int(samples) * 1e-4
