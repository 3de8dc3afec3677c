"""Device memory of the incremental evolve: where its buffers cannot be had the iterations are full
ones, with the same results; and calls that repeat at the same sizes allocate nothing (an allocation
in one context would make every stream of the device wait for it)."""

import ctypes as C

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


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_full_iterations_where_the_buffers_fail(oracle, dtype):
    """After an evolve of full iterations, which has all that one needs, every allocation of an
    incremental evolve on the same context fails in turn."""
    from ridgedetection_amd._lib import OPT_CHAIN, OPT_INJECT_ALLOC_FAILURE
    P = synth.helix3d(20000, seed=4, sigma=0.04, dtype=dtype)
    S0, _ = oracle.choose(P, 0.2)
    ref, iters = oracle.evolve(P, S0, 0.2)
    fixed, _ = oracle.evolve(P, S0, 0.2, 20)
    assert iters > 20
    fell_back = 0
    for k in range(1, 60):
        with _context(dtype) as c:
            c.set_points(P)
            c.set_option(OPT_CHAIN, 2)
            for _ in range(2):
                c.set_chosen(S0)
                np.testing.assert_array_equal(c.evolve(0.2)[0], ref)
            c.set_option(OPT_CHAIN, 1)
            c.set_chosen(S0)
            c.set_option(OPT_INJECT_ALLOC_FAILURE, k)
            try:
                it = C.c_int64()
                c._check(c.lib.rdhip_evolve(c.h, 0.2, 0, C.byref(it)))
            finally:
                c.set_option(OPT_INJECT_ALLOC_FAILURE, 0)
            inc = c.evolve_path()["incremental"]
            print(f"case incremental memory {np.dtype(dtype).name} failing allocation {k}: incremental={inc}",
                  flush=True)
            np.testing.assert_array_equal(c.points(), ref)
            assert it.value == iters
            # the memory is there again: the next call runs incrementally
            c.set_chosen(S0)
            c.evolve_fixed(0.2, 20)
            assert c.evolve_path()["incremental"] > 0
            np.testing.assert_array_equal(c.points(), fixed)
            if inc:
                break
            fell_back += 1
    else:
        pytest.fail("no evolve ran with all of its allocations")
    assert fell_back >= 8


def test_a_batch_falls_back(oracle):
    """The same with several segments: every run either reports the failure or has the oracle's ridges."""
    from ridgedetection_amd._lib import OPT_INJECT_ALLOC_FAILURE, RDError
    clouds = [synth.helix3d(n, seed=60 + i, sigma=0.04) for i, n in enumerate((600, 9000, 513, 4000))]
    radii = [0.2, 0.25, 0.22, 0.3]
    want = [oracle.ridge_detection(p, r, 2 * r)[0] for p, r in zip(clouds, radii)]
    full = 0
    for k in range(1, 200):
        with _context(np.float32) as c:
            c.set_option(OPT_INJECT_ALLOC_FAILURE, k)
            try:
                res = c.batch(clouds, radii, [2 * r for r in radii])
            except RDError as e:
                assert "out of memory" in str(e)
                continue
            finally:
                c.set_option(OPT_INJECT_ALLOC_FAILURE, 0)
            for S, ref in zip(res, want):
                np.testing.assert_array_equal(S, ref)
            again = c.batch(clouds, radii, [2 * r for r in radii])
            for S, ref in zip(again, want):
                np.testing.assert_array_equal(S, ref)
            full += 1
    print(f"case incremental memory batch: {full} runs without an error", flush=True)
    assert full >= 8
