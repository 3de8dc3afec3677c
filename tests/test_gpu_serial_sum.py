"""The ordered sums of long chains (every value of a chain added in sample order, computed in
parallel binade by binade): sums, counts and the evolved points of one iteration against the
oracle's serial sums, bit for bit, for values that cross binades back and forth, land exactly
between two representable sums, stay on a power of two, cancel, or are tiny, at lengths around the
1024- and 2048-value tiles and the length from which a chain is summed by a wave."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KINDS = ["positive", "hover", "halves", "ones", "cancel", "tiny", "mixed_scale", "growing", "negative"]


def _values(kind, n, g, dtype):
    u = g.uniform(0.0, 1.0, n)
    if kind == "positive":
        v = 1.0 + u
    elif kind == "negative":
        v = -3.0 - u
    elif kind == "hover":                      # the running sum wanders around zero
        v = g.normal(0.0, 0.1, n)
    elif kind == "halves":                     # many sums exactly between two representable ones
        v = g.integers(-3, 64, n) * 0.5 + g.integers(0, 2, n) * 2.0 ** (-10 if dtype == np.float32 else -39)
    elif kind == "ones":                       # the sum reaches every power of two exactly
        v = np.ones(n)
    elif kind == "cancel":                     # large values that cancel, small ones between them
        v = np.where(np.arange(n) % 3 == 0, 1.0e4 + u, np.where(np.arange(n) % 3 == 1, -1.0e4 - u, u * 1e-4))
    elif kind == "tiny":
        v = u * (1e-41 if dtype == np.float32 else 1e-320)
    elif kind == "mixed_scale":
        v = g.normal(0.0, 1.0, n) * 10.0 ** g.uniform(-6, 6, n)
    else:
        v = np.exp(np.linspace(-20.0, 12.0, n)) * (0.9 + 0.2 * u)
    return v.astype(dtype)


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("n", [1024, 1025, 1537, 2047, 2048, 2049, 4099, 40001])
def test_one_chain_of_every_kind(oracle, n, dtype):
    from ridgedetection_amd._lib import Context
    g = np.random.Generator(np.random.PCG64(n))
    for a in range(0, len(KINDS), 3):
        kinds = KINDS[a:a + 3]
        P = np.ascontiguousarray(np.stack([_values(k, n, g, dtype) for k in kinds], axis=1))
        S = P[:1].copy()
        r = 1.0e9
        print(f"case serial sum n={n} {np.dtype(dtype).name} {kinds}", flush=True)
        with Context(3, dtype) as c:
            c.set_points(P)
            c.set_chosen(S)
            got, flag, counts, sums, labels, moved = c.evolve_iteration(r)
        ref = oracle.evolve_iter(P, S, r)
        np.testing.assert_array_equal(counts, ref[2])
        assert counts[0] == n
        np.testing.assert_array_equal(sums.view(np.uint8), ref[3].view(np.uint8))
        np.testing.assert_array_equal(got.view(np.uint8), ref[0].view(np.uint8))


@pytest.mark.parametrize("chain", [0, 2])
def test_interleaved_chains(oracle, chain):
    """Several long chains whose members alternate, under both member orderings."""
    from ridgedetection_amd._lib import Context, OPT_CHAIN
    g = np.random.Generator(np.random.PCG64(5))
    n = 30011
    centres = np.array([[0.0, 0.0], [40.0, -40.0], [-0.01, 80.0], [1.0e3, 1.0e3]])
    P = (centres[g.integers(0, 4, n)] + g.normal(0.0, 3.0, (n, 2))).astype(np.float32)
    S = centres.astype(np.float32)
    print(f"case interleaved chains chain={chain}", flush=True)
    with Context(2, np.float32) as c:
        c.set_option(OPT_CHAIN, chain)
        c.set_points(P)
        c.set_chosen(S)
        for _ in range(3):
            got, flag, counts, sums, labels, moved = c.evolve_iteration(30.0)
            ref = oracle.evolve_iter(P, S, 30.0)
            np.testing.assert_array_equal(labels, ref[4])
            np.testing.assert_array_equal(sums, ref[3])
            np.testing.assert_array_equal(got, ref[0])
            S = got
