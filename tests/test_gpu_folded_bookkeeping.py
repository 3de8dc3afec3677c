"""Segments that converge inside a launch batch of incremental iterations, where the bookkeeping of
an iteration runs beside the member scatter of the next: the last block of that launch stores the
done flags while the other blocks read them, so a block's waves may see different values.  Blocks of
several waves, one to many a segment, against the oracle and against full iterations (RDHIP_OPT_CHAIN
2), whose flags change between launches only."""

import numpy as np
import pytest

from ridgedetection_amd import synth

pytestmark = pytest.mark.gpu


def _context(dim, dtype, per_sync, chain=1):
    from ridgedetection_amd._lib import Context, OPT_CHAIN, OPT_ITERS_PER_SYNC, OPT_LOCAL
    c = Context(dim, dtype)
    c.set_option(OPT_LOCAL, 0)
    c.set_option(OPT_CHAIN, chain)
    c.set_option(OPT_ITERS_PER_SYNC, per_sync)
    return c


@pytest.mark.parametrize("per_sync", [8, 64])
@pytest.mark.parametrize("scale", [1, 5], ids=["256-sample-blocks", "1024-sample-blocks"])
def test_many_segments_converge_apart(per_sync, scale):
    clouds, r1 = [], []
    for i in range(60):
        n = (300 + 37 * i) * scale
        clouds.append(synth.spiral2d(n, seed=200 + i) if i % 2 else
                      np.ascontiguousarray(synth.helix3d(n, seed=200 + i, sigma=0.04)[:, :2]))
        r1.append(0.4 + 0.003 * i if i % 2 else 0.1 + 0.002 * i)
    total = sum(len(p) for p in clouds)
    assert total >= 262144 if scale > 1 else total < 131072
    res = []
    for chain in (1, 2):
        print(f"case folded batch per_sync={per_sync} scale={scale} samples={total} chain={chain}", flush=True)
        with _context(2, np.float32, per_sync, chain) as c:
            res.append(c.batch(clouds, r1, [2 * r for r in r1]))
    for i, (a, b) in enumerate(zip(*res)):
        np.testing.assert_array_equal(a, b, err_msg=f"cloud {i}")


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_one_segment_converges_inside_a_batch(oracle, dtype):
    P = synth.spiral2d(9000, seed=12, dtype=dtype)
    S0, _ = oracle.choose(P, 0.45)
    ref, iters = oracle.evolve(P, S0, 0.45)
    for per_sync in (iters - 2, iters - 1, iters, iters + 1, iters + 30):
        print(f"case folded one segment iters={iters} per_sync={per_sync} {np.dtype(dtype).name}", flush=True)
        with _context(2, dtype, per_sync) as c:
            c.set_points(P)
            c.set_chosen(S0)
            S, it = c.evolve(0.45)
        np.testing.assert_array_equal(S, ref)
        assert it == iters
