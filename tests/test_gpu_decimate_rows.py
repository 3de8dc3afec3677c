"""Decimation where neighbour rows are about as long as the provisional rows (32 entries), shorter
and much longer, in orders with and without locality: kept points against the oracle, bit for bit,
both rules."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("rule", [0, 1])
@pytest.mark.parametrize("shuffled", [False, True])
@pytest.mark.parametrize("size", [32, 33, 34, 150])
def test_cluster_sizes(oracle, size, shuffled, rule, dtype):
    from ridgedetection_amd._lib import Context
    g = np.random.Generator(np.random.PCG64(size))
    clusters = 4500 // size
    centres = g.uniform(-5.0, 5.0, (clusters, 4))
    # half of a cluster within r2 of each other, the rest between r2 and 2 r2
    off = g.normal(0.0, 1.0, (clusters, size, 4))
    off *= (g.uniform(0.0, 0.09, (clusters, size)) / np.linalg.norm(off, axis=2))[:, :, None]
    S = (centres[:, None, :] + off).reshape(-1, 4)
    if shuffled:
        S = S[g.permutation(len(S))]
    S = np.ascontiguousarray(S.astype(dtype))
    print(f"case decimate clusters of {size} shuffled={shuffled} rule={rule} {np.dtype(dtype).name}", flush=True)
    with Context(4, dtype) as c:
        c.set_points(S)
        c.set_chosen(S)
        SD, keep = c.decimate(0.1, rule=rule)
    ref, kept = oracle.decimate(S, 0.1, nocopy=rule == 1)
    np.testing.assert_array_equal(np.flatnonzero(keep), kept)
    np.testing.assert_array_equal(SD, ref)


@pytest.mark.parametrize("dim,dtype", [(2, np.float32), (3, np.float64)])
def test_long_rows_of_many_groups(oracle, dim, dtype):
    """Batches decimate per cloud: blocks of 64 elements hold several clouds' points, some with
    rows longer than the provisional ones and some without."""
    from ridgedetection_amd import synth
    from ridgedetection_amd._lib import Context
    g = np.random.Generator(np.random.PCG64(7 + dim))
    clouds = []
    for i in range(24):
        P = synth.segment_chain(int(g.integers(300, 9000)), dim, seed=50 + i, sigma=0.03, dtype=dtype)
        r1 = float(g.uniform(0.04, 0.12))
        clouds.append((P, r1, float(g.uniform(2.0, 8.0)) * r1))
    print(f"case decimate batch d={dim} {np.dtype(dtype).name}", flush=True)
    with Context(dim, dtype) as c:
        res = c.batch([p for p, _, _ in clouds], [a for _, a, _ in clouds], [b for _, _, b in clouds])
    for (P, r1, r2), S in zip(clouds, res):
        np.testing.assert_array_equal(S, oracle.ridge_detection(P, r1, r2)[0])


@pytest.mark.parametrize("rule", [0, 1])
@pytest.mark.parametrize("n", [3, 4, 63, 64, 65, 129, 777, 2047])
def test_walk_in_lds(oracle, n, rule):
    """Groups below 2,048 elements are walked in LDS: the edges of its windows of 64, rows that fit
    and (the dense set of 777 and 2,047) rows that do not, and sets that thin out to three points."""
    from ridgedetection_amd._lib import Context
    g = np.random.Generator(np.random.PCG64(n))
    S = g.uniform(0.0, 1.0, (n, 3)).astype(np.float32)
    for r2 in (0.02, 0.5 / n ** (1 / 3), 1.0 / n ** (1 / 3), 0.4, 3.0):
        print(f"case walk n={n} rule={rule} r2={r2:.4f}", flush=True)
        with Context(3, np.float32) as c:
            c.set_points(S)
            c.set_chosen(S)
            got, keep = c.decimate(r2, rule=rule)
        ref, rkept = oracle.decimate(S, r2, nocopy=rule == 1)
        np.testing.assert_array_equal(got, ref)
        np.testing.assert_array_equal(np.flatnonzero(keep), rkept)
