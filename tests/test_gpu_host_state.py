"""What the host keeps or reads while the device runs: the chosen counts (read back once after each
change) through every call that changes them, and the outcome of evolve batches, one of which may be
in flight past convergence or an iteration limit."""

import numpy as np
import pytest

from ridgedetection_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_counts_follow_every_change(oracle, dtype):
    from ridgedetection_amd._lib import Context
    print(f"case counts {np.dtype(dtype).name}", flush=True)
    with Context(2, dtype) as c:
        for n, r in ((3000, 0.45), (7001, 0.6), (1, 0.5), (2500, 0.3)):
            P = synth.spiral2d(n, seed=n, dtype=dtype)
            c.set_points(P)
            S0, idx = c.choose(r)
            ref, ridx = oracle.choose(P, r)
            np.testing.assert_array_equal(S0, ref)
            half = np.ascontiguousarray(ref[::2])
            c.set_chosen(half)
            np.testing.assert_array_equal(c.points(), half)
            got, flag, counts, sums, labels, moved = c.evolve_iteration(r)
            want = oracle.evolve_iter(P, half, r)
            np.testing.assert_array_equal(got, want[0])
            np.testing.assert_array_equal(counts, want[2])
            np.testing.assert_array_equal(sums, want[3])
            np.testing.assert_array_equal(labels, want[4])
            kept, keep = c.decimate(2 * r)
            np.testing.assert_array_equal(c.points(), kept)
            assert len(kept) == int(np.count_nonzero(keep))
            S, it = c.evolve(r)
            ref, rit = oracle.evolve(P, kept, r)
            np.testing.assert_array_equal(S, ref)
            assert it == rit


def test_limits_while_a_batch_is_in_flight(oracle):
    from ridgedetection_amd._lib import Context, OPT_EVOLVE_GUARD, OPT_LOCAL
    P = synth.helix3d(20000, seed=4, sigma=0.04)
    S0, _ = oracle.choose(P, 0.2)
    for cap in (39, 40, 41, 48, 49, 56, 57):
        print(f"case limits cap={cap}", flush=True)
        with Context(3, np.float32) as c:
            c.set_option(OPT_LOCAL, 0)
            c.set_points(P)
            c.set_chosen(S0)
            S, it = c.evolve(0.2, cap)
            ref, rit = oracle.evolve(P, S0, 0.2, cap)
            np.testing.assert_array_equal(S, ref)
            assert it == rit
            c.set_chosen(S0)
            c.set_option(OPT_EVOLVE_GUARD, 48)
            if rit >= 48:
                with pytest.raises(Exception, match="iteration guard"):
                    c.evolve(0.2, 0)
