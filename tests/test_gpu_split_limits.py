"""Work items cut while the slots of their sub-items are scarce ("split_parts"): which items are cut may
depend on the lists alone, not on the order in which wavefronts ask for slots, so that a solve repeated
on the same inputs gives the same bits.  Against the same solve without cuts the tolerance of
test_gpu_split.py (FP64 sums in another order) holds in FP64; in the mixed form list ranges regroup FP32
partials, 15 u of a sum of positive terms each: 1e-6."""
import numpy as np
import pytest

from cosmosphere_amd import Library
from gpu_common import DEFAULT_ITEMS, dataset, gpu_run, rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _reset_options():
    yield
    for kernel in ("cubic", "quintic"):
        lib = Library(kernel)
        for k, v in dict(DEFAULT_ITEMS, split_parts=0).items():
            lib.set_option(k, v)


@pytest.mark.parametrize("split_len", [-1, 8])
@pytest.mark.parametrize("parts", [2, 70, 700, 0])
@pytest.mark.parametrize("mapping", [0, 1, 2])
@pytest.mark.parametrize("precision", [0, 1])
def test_same_bits_again(precision, mapping, parts, split_len):
    c = dataset("plummer_quintic")
    opts = dict(precision=precision, gradients=False, mapping=mapping, units=1)
    print("case limits", precision, mapping, parts, split_len, flush=True)
    lib, whole = gpu_run(c, split_len=0, split_parts=0, **opts)
    ref = {k: lib.array(k).copy() for k in ("h", "rho")}
    first = None
    for _ in range(4):
        lib, iters = gpu_run(c, split_len=split_len, split_parts=parts, **opts)
        got = {k: lib.array(k).copy() for k in ("h", "rho", "gradh")}
        split = lib.passes()[:, 13].copy()
        if parts:
            assert (2 * split <= parts).all()            # two sub-items each, at least
        if first is None:
            first = got, split, iters
            continue
        assert iters == first[2] and np.array_equal(split, first[1])
        for k, v in first[0].items():
            assert np.array_equal(got[k], v), k
    assert first[2] == whole
    for k, v in ref.items():
        assert rel_err(first[0][k], v) < (1e-11 if precision == 0 else 1e-6), k
