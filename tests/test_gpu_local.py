"""Segment-local evolve with the samples in LDS (samples compared with the moved points only, chains
whose members changed summed only): evolved points and iteration counts against the oracle, bit for
bit, around the block's 1024 threads and waves, where a segment just fits or just does not fit the
LDS, for every dimension and both value types, with caps, equal, infinite and NaN samples."""

import numpy as np
import pytest

from ridgedetection_amd import synth

pytestmark = pytest.mark.gpu


def _check(oracle, P, r, caps=(0,), S0=None):
    from ridgedetection_amd._lib import Context
    if S0 is None:
        S0, _ = oracle.choose(P, r)
    print(f"case local n={len(P)} d={P.shape[1]} {P.dtype.name} K={len(S0)}", flush=True)
    with Context(P.shape[1], P.dtype) as c:
        c.set_points(P)
        for cap in caps:
            c.set_chosen(S0)
            S, it = c.evolve(r, cap)
            ref, rit = oracle.evolve(P, S0, r, cap)
            np.testing.assert_array_equal(S, ref)
            assert it == rit


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1024, 1025, 2048, 2100, 3500, 4600, 8192, 8193])
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_sizes_and_caps(oracle, n, dtype):
    _check(oracle, synth.spiral2d(n, seed=n, dtype=dtype), 0.45, caps=(1, 2, 3, 7, 0))


@pytest.mark.parametrize("dim", list(range(1, 13)))
def test_dimensions(oracle, dim):
    for n, dtype in ((1500, np.float64), (900, np.float32)):
        P = synth.segment_chain(n, dim, seed=dim, sigma=0.03, segments=6, dtype=dtype)
        _check(oracle, P, 0.02 if dim == 1 else 0.08 * np.sqrt(dim))


@pytest.mark.parametrize("K", [1, 16, 63, 64, 65, 1008, 1024])
def test_chosen_counts(oracle, K):
    """One chain of every sample up to the most chosen points the path takes."""
    P = synth.helix3d(1500, seed=K)
    _check(oracle, P, 0.4, S0=np.ascontiguousarray(P[:K]))


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_unusual_samples(oracle, dtype):
    P = synth.helix3d(1700, seed=3, dtype=dtype)
    S0, _ = oracle.choose(P, 0.3)
    P[5::97, 1] = np.nan
    P[11::101, 0] = np.inf
    P[17::103, 2] = -np.inf
    P[3::50] = P[4::50]
    _check(oracle, P, 0.3, S0=S0)
    g = np.arange(32, dtype=dtype)           # equal distances everywhere: the first index decides
    L = np.ascontiguousarray(np.stack(np.meshgrid(g, g), axis=-1).reshape(-1, 2))
    _check(oracle, L, 3.0, S0=np.ascontiguousarray(L[(L[:, 0] % 4 == 0) & (L[:, 1] % 4 == 2)]))


def test_tiles_and_batches(oracle):
    from ridgedetection_amd._lib import Context
    P = synth.segment_chain(30000, 4, seed=8, sigma=0.03, dtype=np.float64)
    print("case local tiles and batch", flush=True)
    with Context(4, np.float64) as c:
        c.set_points(P)
        for alg in (0, 6):
            np.testing.assert_array_equal(c.tiled(alg, 0.12, 0.24, 1000, [3] * 4),
                                          oracle.tiled(alg, P, 0.12, 0.24, 1000, [3] * 4))
        clouds = [np.ascontiguousarray(synth.segment_chain(n, 4, seed=n, sigma=0.05, dtype=np.float64))
                  for n in (300, 1700, 1, 900, 2049, 64)]
        res = c.batch(clouds, [0.3] * 6, [0.6] * 6)
    for Q, S in zip(clouds, res):
        np.testing.assert_array_equal(S, oracle.ridge_detection(Q, 0.3, 0.6)[0])
