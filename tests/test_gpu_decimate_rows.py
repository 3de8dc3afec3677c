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
