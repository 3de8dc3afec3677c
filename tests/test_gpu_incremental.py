"""Incremental evolve iterations (samples in spatial blocks that look only at the chosen points
within reach, and only when one of those moved; chains whose members did not change keep their
sums): evolved points and iteration counts against the oracle, bit for bit, at the edges of the
blocks, for every dimension, both value types, several segments, caps that stop early, equal,
infinite and NaN samples; and against the full iterations (RDHIP_OPT_CHAIN 2)."""

import numpy as np
import pytest

from ridgedetection_amd import synth

pytestmark = pytest.mark.gpu


def _ctx(dim, dtype, chain=1):
    from ridgedetection_amd._lib import Context, OPT_CHAIN, OPT_LOCAL
    c = Context(dim, dtype)
    c.set_option(OPT_LOCAL, 0)   # small clouds too
    c.set_option(OPT_CHAIN, chain)
    return c


def _evolve_check(oracle, P, r, caps=(0,)):
    S0, _ = oracle.choose(P, r)
    print(f"case incremental n={len(P)} d={P.shape[1]} {P.dtype.name} K={len(S0)}", flush=True)
    with _ctx(P.shape[1], P.dtype) as c:
        c.set_points(P)
        for cap in caps:
            c.set_chosen(S0)
            S, it = c.evolve(r, cap)
            ref, rit = oracle.evolve(P, S0, r, cap)
            np.testing.assert_array_equal(S, ref)
            assert it == rit
    return len(S0)


@pytest.mark.parametrize("n", [511, 512, 513, 1023, 4096, 4609, 20000])
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_block_edges_and_caps(oracle, n, dtype):
    P = synth.spiral2d(n, seed=n, dtype=dtype)
    K = _evolve_check(oracle, P, 0.45, caps=(4, 5, 9, 17, 0))
    assert K >= 48


@pytest.mark.parametrize("dim", list(range(1, 13)))
def test_dimensions(oracle, dim):
    dtype = np.float32 if dim % 2 else np.float64
    P = synth.segment_chain(9000, dim, seed=dim, sigma=0.03, segments=6, dtype=dtype)
    r = 0.02 if dim == 1 else 0.06 * np.sqrt(dim)
    K = _evolve_check(oracle, P, r)
    assert K >= 48


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_unusual_samples(oracle, dtype):
    P = synth.helix3d(12000, seed=3, dtype=dtype)
    P[5::97, 1] = np.nan
    P[11::101, 0] = np.inf
    P[17::103, 2] = -np.inf
    P[3::50] = P[4::50]                      # equal samples
    P[:3] = P[100]
    Q = P[np.isfinite(P).all(1)]
    S0, _ = oracle.choose(np.ascontiguousarray(Q), 0.2)
    print("case incremental NaN and infinite samples", flush=True)
    with _ctx(3, dtype) as c:
        c.set_points(P)
        c.set_chosen(S0)
        S, it = c.evolve(0.2)
    ref, rit = oracle.evolve(P, S0, 0.2)
    np.testing.assert_array_equal(S, ref)
    assert it == rit


def test_grid_ties(oracle):
    """Samples and chosen points on a lattice: equal distances everywhere, so the first index
    decides."""
    g = np.arange(64, dtype=np.float32)
    P = np.stack(np.meshgrid(g, g), axis=-1).reshape(-1, 2)
    P = np.ascontiguousarray(P[np.random.Generator(np.random.PCG64(1)).permutation(len(P))])
    S0 = np.ascontiguousarray(P[(P[:, 0] % 4 == 0) & (P[:, 1] % 4 == 2)])
    print(f"case incremental lattice K={len(S0)}", flush=True)
    for r in (2.0, 3.0, 50.0):
        with _ctx(2, np.float32) as c:
            c.set_points(P)
            c.set_chosen(S0)
            S, it = c.evolve(r, 30)
        ref, rit = oracle.evolve(P, S0, r, 30)
        np.testing.assert_array_equal(S, ref)
        assert it == rit


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_fixed_iterations_match_full_ones(dtype):
    """evolve_fixed past convergence, repeated calls, new points and new chosen sets on one context."""
    print(f"case incremental fixed iterations {np.dtype(dtype).name}", flush=True)
    res = {}
    for chain in (1, 2):
        out = []
        with _ctx(3, dtype, chain) as c:
            for seed in (5, 6):
                c.set_points(synth.helix3d(50001 - seed, seed=seed, dtype=dtype))
                S0, _ = c.choose(0.2)
                for iters in (4, 13, 30):
                    c.evolve_fixed(0.2, iters)
                    out.append(c.points())
                c.set_chosen(S0[::2].copy())
                c.evolve_fixed(0.21, 12)
                out.append(c.points())
        res[chain] = out
    for a, b in zip(res[1], res[2]):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("dim,dtype", [(2, np.float32), (3, np.float64)])
def test_batches(oracle, dim, dtype):
    clouds = []
    for i, n in enumerate([600, 20000, 513, 9000, 1, 30001, 512, 7000]):
        P = synth.helix3d(n, seed=60 + i, sigma=0.04, dtype=dtype)[:, :dim]
        clouds.append((np.ascontiguousarray(P), 0.1 + 0.01 * i))
    print(f"case incremental batch d={dim} {np.dtype(dtype).name}", flush=True)
    with _ctx(dim, dtype) as c:
        res = c.batch([p for p, _ in clouds], [r for _, r in clouds], [2 * r for _, r in clouds])
        again = c.batch([p for p, _ in clouds], [r for _, r in clouds], [2 * r for _, r in clouds])
    for (P, r), S, S2 in zip(clouds, res, again):
        ref, _ = oracle.ridge_detection(P, r, 2 * r)
        np.testing.assert_array_equal(S, ref)
        np.testing.assert_array_equal(S2, ref)


@pytest.mark.parametrize("alg", [0, 1, 6])
def test_tiles(oracle, alg):
    P = synth.helix3d(40000, seed=33)
    print(f"case incremental tiles alg={alg}", flush=True)
    with _ctx(3, np.float32) as c:
        c.set_points(P)
        S = c.tiled(alg, 0.06, 0.12, 20000, [2, 2, 2])
    np.testing.assert_array_equal(S, oracle.tiled(alg, P, 0.06, 0.12, 20000, [2, 2, 2]))


@pytest.mark.parametrize("per_sync", [1, 2, 8])
def test_caps_around_launch_batches(oracle, per_sync):
    """The bookkeeping of an iteration runs inside the next one of its launch batch: caps that end
    on either side of a batch's first and last iteration, several segments that converge apart."""
    from ridgedetection_amd._lib import OPT_ITERS_PER_SYNC
    P = synth.spiral2d(6000, seed=9)
    S0, _ = oracle.choose(P, 0.45)
    clouds = [synth.spiral2d(n, seed=n) for n in (900, 6000, 2500)]
    radii = [0.45, 0.5, 0.55]
    for cap in (1, 2, 3, 7, 8, 9, 10, 16, 17, 18):
        print(f"case incremental cap={cap} per_sync={per_sync}", flush=True)
        with _ctx(2, np.float32) as c:
            c.set_option(OPT_ITERS_PER_SYNC, per_sync)
            c.set_points(P)
            c.set_chosen(S0)
            S, it = c.evolve(0.45, cap)
            res = c.batch(clouds, radii, [2 * r for r in radii], max_evolve_iters=cap)
        ref, rit = oracle.evolve(P, S0, 0.45, cap)
        np.testing.assert_array_equal(S, ref)
        assert it == rit
        for got, cloud, r in zip(res, clouds, radii):
            np.testing.assert_array_equal(got, oracle.ridge_detection(cloud, r, 2 * r, max_evolve_iter=cap)[0])


def test_large_count_tables():
    """More than 4 MB of counts: eight full iterations come first."""
    from ridgedetection_amd._lib import OPT_AUTOTUNE
    P = synth.helix3d(700000, seed=21, sigma=0.03)
    res = []
    for auto in (1, 0):
        with _ctx(3, np.float32) as c:
            c.set_option(OPT_AUTOTUNE, auto)
            c.set_points(P)
            S0, _ = c.choose(0.08)
            print(f"case incremental large counts K={len(S0)} autotune={auto}", flush=True)
            assert 1600 < len(S0) <= 2048
            c.evolve_fixed(0.08, 13)
            res.append(c.points())
            S, it = c.evolve(0.08, 21)
            res.append(S)
    np.testing.assert_array_equal(res[0], res[2])
    np.testing.assert_array_equal(res[1], res[3])
