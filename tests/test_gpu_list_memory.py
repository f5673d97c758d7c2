"""The slots of tokens that lists keep between their count and their fill are as long as memory allows: where
the longer ones are refused ("alloc_limit" stands for a card that is nearly full), shorter ones serve, with
the same results bit for bit, and the solve does not fail.  The plan of captured launches holds the
slot length: a solve after a change of it, at the same sizes, uses the new one."""
import numpy as np
import pytest

from cosmosphere_amd import Library
from gpu_common import DEFAULT_ITEMS, dataset, gpu_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["plummer_quintic", "plummer_cubic"])
def test_shorter_slots(name):
    c = dataset(name)
    lib = Library(c["kernel"])
    try:
        out = []
        cap = 2048 + 1      # leaves, rounded up (20,000 particles: 1,025 to 2,048 leaves), and one
        for limit, slots in ((0, 2048), (cap * 4 * 1024 * 9 // 8 + 256, 1024), (cap * 4 * 300, 256), (0, 2048)):
            print("case memory", name, limit, flush=True)
            lib.set_option("alloc_limit", limit)
            gpu_run(c, split_len=0)
            assert 1024 < lib.stat("n_leaves") <= 2048
            assert lib.stat("list_slot_tokens") == slots
            out.append([lib.array(k).copy() for k in ("h", "rho", "gradh")] + [lib.passes()[:, 10].copy()])
        for other in out[1:]:
            for a, b in zip(out[0], other):
                assert np.array_equal(a, b)
    finally:
        lib.set_option("alloc_limit", 0)
        for k, v in DEFAULT_ITEMS.items():
            lib.set_option(k, v)
