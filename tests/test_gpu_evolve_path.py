"""Which form an evolve ran in (rdhip_evolve_path): incremental iterations under the default
options only, the segment-local kernel with its samples in LDS where they fit; and the iteration guard
while a launch batch is in flight beyond the one whose outcome is known."""

import numpy as np
import pytest

from ridgedetection_amd import synth

pytestmark = pytest.mark.gpu


def _evolve_all(c, P, S0, r):
    """incremental after each of the two evolve calls, and the evolved points"""
    c.set_points(P)
    c.set_chosen(S0)
    S, _ = c.evolve(r)
    seen = [c.evolve_path()["incremental"]]
    c.set_chosen(S0)
    c.evolve_fixed(r, 9)
    return seen + [c.evolve_path()["incremental"]], S


@pytest.mark.parametrize("dim", [1, 2, 3, 6, 12])
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_default_options_run_incrementally(oracle, dim, dtype):
    from ridgedetection_amd._lib import Context, OPT_AUTOTUNE, OPT_CHAIN, OPT_LOCAL, OPT_SCREEN, OPT_SUM_MODE
    P = synth.segment_chain(9000, dim, seed=dim, sigma=0.03, segments=6, dtype=dtype)
    r = 0.02 if dim == 1 else 0.06 * np.sqrt(dim)
    S0, _ = oracle.choose(P, r)
    ref, _ = oracle.evolve(P, S0, r)
    assert 8 <= len(S0) <= 2048
    for opts, inc in (({}, True), ({OPT_CHAIN: 2}, False), ({OPT_CHAIN: 0}, False), ({OPT_AUTOTUNE: 0}, False),
                      ({OPT_SCREEN: 1}, False), ({OPT_SUM_MODE: 1}, False)):
        print(f"case path d={dim} {np.dtype(dtype).name} K={len(S0)} options={opts}", flush=True)
        with Context(dim, dtype) as c:
            c.set_option(OPT_LOCAL, 0)
            for o, v in opts.items():
                c.set_option(o, v)
            seen, S = _evolve_all(c, P, S0, r)
        assert [s > 0 for s in seen] == [inc, inc]
        if OPT_SUM_MODE not in opts:
            np.testing.assert_array_equal(S, ref)


def test_few_and_many_chosen_points_run_in_full(oracle):
    from ridgedetection_amd._lib import Context, OPT_LOCAL
    P = synth.helix3d(30000, seed=2, sigma=0.04)
    for K, inc in ((7, False), (8, True), (2048, True), (2049, False)):
        print(f"case path K={K}", flush=True)
        with Context(3, np.float32) as c:
            c.set_option(OPT_LOCAL, 0)
            c.set_points(P)
            c.set_chosen(np.ascontiguousarray(P[:K]))
            S, it = c.evolve(0.2, 12)
            assert (c.evolve_path()["incremental"] > 0) == inc
        ref, rit = oracle.evolve(P, np.ascontiguousarray(P[:K]), 0.2, 12)
        np.testing.assert_array_equal(S, ref)
        assert it == rit


@pytest.mark.parametrize("n,segments", [(500, 1), (2000, 1), (8192, 0), (9000, 0)])
def test_local_samples_in_lds(oracle, n, segments):
    """8192 samples of three doubles with their distances are 256 KB, more than a workgroup has."""
    from ridgedetection_amd._lib import Context
    P = synth.helix3d(n, seed=n, sigma=0.04, dtype=np.float64)
    S0, _ = oracle.choose(P, 0.25)
    print(f"case path local n={n} K={len(S0)}", flush=True)
    with Context(3, np.float64) as c:
        c.set_points(P)
        c.set_chosen(S0)
        S, it = c.evolve(0.25)
        t = c.evolve_path()
    assert (t["local_lds"], t["incremental"]) == (segments, 0)
    ref, rit = oracle.evolve(P, S0, 0.25)
    np.testing.assert_array_equal(S, ref)
    assert it == rit


@pytest.mark.parametrize("guard", [41, 60])
def test_guard_with_a_batch_in_flight(oracle, guard):
    """From the fifth launch on, a batch is in flight beyond the known outcome until three batches
    before the guard: with two iterations a launch that is most of them."""
    from ridgedetection_amd._lib import Context, OPT_EVOLVE_GUARD, OPT_ITERS_PER_SYNC, OPT_LOCAL, RDError
    P = synth.spiral2d(20000, seed=4)
    S0, _ = oracle.choose(P, 0.45)
    ref, iters = oracle.evolve(P, S0, 0.45)
    assert iters > 62
    print(f"case guard={guard} of {iters} iterations", flush=True)
    with Context(2, np.float32) as c:
        c.set_option(OPT_LOCAL, 0)
        c.set_option(OPT_ITERS_PER_SYNC, 2)
        c.set_points(P)
        c.set_chosen(S0)
        c.set_option(OPT_EVOLVE_GUARD, guard)
        with pytest.raises(RDError, match="iteration guard"):
            c.evolve(0.45)
        c.set_option(OPT_EVOLVE_GUARD, 0)
        S, rest = c.evolve(0.45)   # from where the guard stopped it
        np.testing.assert_array_equal(S, ref)
        assert iters - guard - 2 <= rest <= iters - guard + 1
        c.set_chosen(S0)
        S, it = c.evolve(0.45)
    np.testing.assert_array_equal(S, ref)
    assert it == iters


def test_full_iterations_follow_the_current_count_table():
    """A large chosen set (count tables over 4 MB) starts with eight full iterations; a small one on
    the same context afterwards with one, as it would on a context of its own."""
    from ridgedetection_amd._lib import Context
    P = synth.helix3d(1200000, seed=21, sigma=0.03)
    with Context(3, np.float32) as c:
        c.set_points(P)
        S0 = np.ascontiguousarray(c.choose(0.07)[0][:2000])
        assert len(S0) == 2000   # x 586 columns of 2048 samples: 4.7 MB of counts
        for S, full in ((S0, 8), (np.ascontiguousarray(S0[::8]), 1), (S0, 8)):
            c.set_chosen(S)
            c.evolve_fixed(0.08, 12)
            print(f"case path K={len(S)} {c.evolve_path()}", flush=True)
            assert c.evolve_path()["incremental"] == full


@pytest.mark.parametrize("per_sync,guard", [(64, 64), (1, 1), (2, 3), (5, 16), (8, 8)])
def test_guard_stops_after_whole_launch_batches(oracle, per_sync, guard):
    """The iteration limit is looked at after every per_sync iterations from the first on."""
    from ridgedetection_amd._lib import Context, OPT_EVOLVE_GUARD, OPT_ITERS_PER_SYNC, OPT_LOCAL, RDError
    P = synth.spiral2d(20000, seed=4)
    S0, _ = oracle.choose(P, 0.45)
    _, iters = oracle.evolve(P, S0, 0.45)
    assert iters == 65
    ran = -(-guard // per_sync) * per_sync
    print(f"case guard={guard} per_sync={per_sync} stops after {ran}", flush=True)
    with Context(2, np.float32) as c:
        c.set_option(OPT_LOCAL, 0)
        c.set_option(OPT_ITERS_PER_SYNC, per_sync)
        c.set_points(P)
        c.set_chosen(S0)
        c.set_option(OPT_EVOLVE_GUARD, guard)
        with pytest.raises(RDError, match="iteration guard"):
            c.evolve(0.45)
        np.testing.assert_array_equal(c.points(), oracle.evolve(P, S0, 0.45, ran)[0])


def test_guard_within_the_full_iterations():
    """Eight full iterations first, stopped after three of them."""
    from ridgedetection_amd._lib import Context, OPT_EVOLVE_GUARD, OPT_ITERS_PER_SYNC, RDError
    P = synth.helix3d(1200000, seed=21, sigma=0.03)
    with Context(3, np.float32) as c:
        c.set_points(P)
        S0 = np.ascontiguousarray(c.choose(0.07)[0][:2000])
        c.set_chosen(S0)
        want, _ = c.evolve(0.07, 3)
        c.set_chosen(S0)
        c.set_option(OPT_ITERS_PER_SYNC, 3)
        c.set_option(OPT_EVOLVE_GUARD, 2)
        print(f"case guard within {len(S0)} chosen points' full iterations", flush=True)
        with pytest.raises(RDError, match="iteration guard"):
            c.evolve(0.07)
        assert c.evolve_path()["incremental"] == 8
        np.testing.assert_array_equal(c.points(), want)


def test_short_evolves_on_new_points(oracle):
    """Ordering new samples by space pays from eight iterations on, or from four where a full scan
    has 2^26 pairs or more; an order that is there is used."""
    from ridgedetection_amd._lib import Context, OPT_LOCAL
    for n, steps in ((20000, ((7, 0), (8, 1), (4, 1), (1, 1))), (400000, ((3, 0), (4, 1), (2, 1)))):
        P = synth.helix3d(n, seed=4, sigma=0.04)
        with Context(3, np.float32) as c:
            c.set_option(OPT_LOCAL, 0)
            c.set_points(P)
            S0, _ = c.choose(0.2)
            for iters, inc in steps:
                c.set_chosen(S0)
                c.evolve_fixed(0.2, iters)
                print(f"case path n={n} K={len(S0)} iterations={iters} {c.evolve_path()}", flush=True)
                assert c.evolve_path()["incremental"] == inc
                if n < 100000:
                    np.testing.assert_array_equal(c.points(), oracle.evolve(P, S0, 0.2, iters)[0])
