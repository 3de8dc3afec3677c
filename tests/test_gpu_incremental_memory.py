"""Device memory of the incremental evolve: where its buffers cannot be had the iterations are full
ones, with the same results; and calls that repeat at the same sizes allocate nothing (an allocation
in one context would make every stream of the device wait for it)."""

import numpy as np
import pytest

from ridgedetection_amd import synth

pytestmark = pytest.mark.gpu


def _context(dtype):
    from ridgedetection_amd._lib import Context, OPT_LOCAL
    c = Context(3, dtype)
    c.set_option(OPT_LOCAL, 0)
    return c


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_repeated_calls_allocate_nothing(oracle, dtype):
    """The next allocation would fail: incremental iterations on new points of the same number and one
    recorded iteration with all of its outputs go through without one."""
    from ridgedetection_amd._lib import OPT_INJECT_ALLOC_FAILURE, _ptr
    r = 0.2
    n, K = 20000, 150
    labels, counts = np.empty(n, np.int32), np.empty(K, np.int32)
    sums, moved = np.empty((K, 3), dtype), np.empty(K, np.uint16)
    with _context(dtype) as c:
        for turn in range(3):
            P = synth.helix3d(n, seed=4 + turn, sigma=0.04, dtype=dtype)
            S0 = np.ascontiguousarray(oracle.choose(P, r)[0][:K])
            print(f"case incremental allocations turn={turn} {np.dtype(dtype).name}", flush=True)
            c.set_points(P)
            c.set_chosen(S0)
            for call in (lambda: c.evolve_fixed(r, 12),
                         lambda: c._check(c.lib.rdhip_evolve_iteration(c.h, r, _ptr(labels), _ptr(counts), _ptr(sums),
                                                                       _ptr(moved), None))):
                c.set_option(OPT_INJECT_ALLOC_FAILURE, 1 if turn else 0)
                try:
                    call()
                finally:
                    c.set_option(OPT_INJECT_ALLOC_FAILURE, 0)
            assert c.evolve_path()["incremental"] == 1
            want = oracle.evolve_iter(P, oracle.evolve(P, S0, r, 12)[0], r)
            np.testing.assert_array_equal(c.points(), want[0])
            np.testing.assert_array_equal(counts, want[2])
            np.testing.assert_array_equal(sums, want[3])
            np.testing.assert_array_equal(labels, want[4])
