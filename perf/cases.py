"""Timed workloads of the ridge-detection library, through its public entry points.

A case is one pass a user's program makes over inputs it already holds: a whole ridge
detection (brute force, tiled, batched), or one phase of it driven by the caller (choose,
evolve, one evolve iteration with its outputs, decimate, the differentiated evolve).

    listed()             the fixed cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  inputs from the seed, resident on the GPU, and the context
    run(state)           one pass; returns all of its outputs
    work(case)           bytes and operations no implementation of the pass can avoid
    exact(case, seed)    the pass in 64-bit arithmetic where it has such a value
"""

from __future__ import annotations

import math

import numpy as np
import torch

from ridgedetection_amd import synth
from ridgedetection_amd._lib import DECIMATE, DECIMATE_NO_COPY, Context


# ---------------------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------------------
def listed():
    return [
        # the smallest interactive call: a scanned outline of 2,000 points in double precision,
        # chosen, evolved and decimated to its ridge; every launch and synchronisation shows
        dict(name="ridge_spiral_2k_f64", kind="ridge", shape="spiral", n=2000, dim=2, dtype="f64",
             sigma=0.1, r=0.45, cap=100),
        # the plain method at its documented size: 20,000 points of an Archimedean spiral
        dict(name="ridge_spiral_20k", kind="ridge", shape="spiral", n=20000, dim=2, dtype="f32",
             sigma=0.1, r=0.45, cap=100),
        # a whole brute-force ridge detection of a large 3-D cloud
        dict(name="ridge_helix_1m", kind="ridge", shape="helix", n=1000000, dim=3, dtype="f32",
             sigma=0.05, r=0.2, cap=0),
        # a caller-driven evolve (the device facade with a fixed iteration count): the phase that
        # dominates brute-force runs
        dict(name="evolve_helix_1m", kind="evolve", shape="helix", n=1000000, dim=3, dtype="f32",
             sigma=0.05, r=0.2, iters=20),
        # one evolve iteration with all of its outputs (labels, counts, sums, moved coordinates)
        # in double precision, five dimensions and a ragged size: a custom driver's inner step
        dict(name="iteration_chain_150k_5d_f64", kind="iteration", shape="chain", n=150001, dim=5,
             dtype="f64", sigma=0.05, r=0.2),
        # a greedy ball cover of scattered high-dimensional data: many chosen points
        dict(name="choose_bezier_200k_6d", kind="choose", shape="bezier", n=200000, dim=6, dtype="f32",
             sigma=0.02, r=0.08),
        # the global decimation a tiled or hand-written driver runs over all chosen points
        dict(name="decimate_bezier_300k_6d", kind="decimate", shape="bezier", n=300000, dim=6, dtype="f32",
             sigma=0.02, r=0.08, no_copy=True),
        # tiled ridge detection, a whole detection per extended tile of the 1M-point helix
        dict(name="tiled_helix_extended_1m", kind="tiled", shape="helix", n=1000000, dim=3, dtype="f32",
             sigma=0.05, r=0.2, algorithm=6, tiles=8, capacity=10000, refine=False),
        # the largest tiled run: 2M points in six dimensions, evolve over own and neighbour tiles
        dict(name="tiled_bezier_grouped_2m_6d", kind="tiled", shape="bezier", n=2000000, dim=6, dtype="f32",
             sigma=0.02, r=0.08, algorithm=1, tiles=4, capacity=10000, refine=False),
        # small tiles in double precision with the end-phase refinement over the whole cloud
        dict(name="tiled_chain_local_120k_4d_f64", kind="tiled", shape="chain", n=120007, dim=4, dtype="f64",
             sigma=0.03, r=0.12, algorithm=0, tiles=3, capacity=2000, refine=True),
        # many uneven clouds of two and three dimensions in one batch
        dict(name="batch_128_mixed", kind="batch", clouds=128, lo=2000, hi=300000, dim=3, dtype="f32", cap=0),
        # the differentiated evolve: forward with checkpoints, then the vector-Jacobian product
        dict(name="vjp_helix_200k", kind="vjp", shape="helix", n=200000, dim=3, dtype="f32",
             sigma=0.05, r=0.2, iters=20, every=4),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["ridge", "ridge", "evolve", "iteration", "choose", "decimate", "tiled", "tiled", "batch",
                       "vjp"])
    dtype = rng.choice(["f32", "f32", "f64"])
    if kind == "batch":
        return dict(kind="batch", clouds=rng.randint(3, 100), lo=1000, hi=_logint(rng, 8000, 200000),
                    dim=rng.choice([2, 3]), dtype=dtype, cap=200)
    shape = rng.choice(["spiral", "helix", "chain", "bezier"])
    c = dict(kind=kind, shape=shape, dtype=dtype)
    c["dim"] = {"spiral": 2, "helix": 3}.get(shape) or rng.randint(2, 6)
    # noise and radius as fractions of the shape's extent (spiral about 18, the others 2 to 5)
    unit = {"spiral": 4.0, "helix": 1.0, "chain": 0.6, "bezier": 0.4}[shape]
    c["sigma"] = round(rng.uniform(0.025, 0.06) * unit, 4)
    c["r"] = round(c["sigma"] * rng.uniform(3.5, 4.5), 4)
    if kind == "ridge":
        c["n"] = _logint(rng, 500, 1000000 if shape != "bezier" else 60000)
        c["cap"] = 100
    elif kind == "evolve":
        c["n"] = _logint(rng, 5000, 1000000 if shape != "bezier" else 200000)
        c["iters"] = rng.randint(3, 24)
    elif kind == "iteration":
        c["n"] = _logint(rng, 2000, 300000)
    elif kind == "choose":
        c["n"] = _logint(rng, 2000, 1000000 if shape != "bezier" else 200000)
    elif kind == "decimate":
        c["n"] = _logint(rng, 5000, 300000)
        c["no_copy"] = rng.random() < 0.5
    elif kind == "tiled":
        c["n"] = _logint(rng, 20000, 1000000)
        c["algorithm"] = rng.choice([0, 1, 2, 4, 5, 6])
        c["tiles"] = 8 if c["dim"] <= 3 else 4 if c["dim"] <= 4 else 3
        c["capacity"] = rng.choice([1000, 4000, 10000])
        c["refine"] = rng.random() < 0.25
    else:
        c["n"] = _logint(rng, 5000, 400000)
        c["iters"] = rng.randint(4, 24)
        c["every"] = rng.choice([0, 3, 4, 8])
    return c


# ---------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------
def _dtype(case):
    return np.float32 if case["dtype"] == "f32" else np.float64


def _cloud(case, seed):
    n, dim, s, dt = case["n"], case["dim"], case["sigma"], _dtype(case)
    if case["shape"] == "spiral":
        return synth.spiral2d(n, seed=seed, sigma=s, dtype=dt)
    if case["shape"] == "helix":
        return synth.helix3d(n, seed=seed, sigma=s, dtype=dt)
    if case["shape"] == "chain":
        return synth.segment_chain(n, dim, seed=seed, sigma=s, dtype=dt)
    return _bezier(n, dim, seed, s, dt)


def _bezier(n, dim, seed, sigma, dt):
    """The distribution of synth.bezier_union (four cubic Bezier curves, 5% uniform outliers,
    shuffled), drawn in the output type so that millions of points take well under a second."""
    g = np.random.Generator(np.random.PCG64(seed))
    ctrl = g.uniform(-1.0, 1.0, (4, 4, dim))
    n_out = n // 20
    which = g.integers(0, 4, n - n_out)
    u = g.random(n - n_out, dtype=np.float32).astype(dt)
    w = np.stack([(1 - u) ** 3, 3 * (1 - u) ** 2 * u, 3 * (1 - u) * u ** 2, u ** 3], axis=1)
    P = np.empty((n, dim), dtype=dt)
    for k in range(4):
        m = np.flatnonzero(which == k)
        P[m] = w[m] @ ctrl[k].astype(dt)
    P[:n - n_out] += g.standard_normal((n - n_out, dim), dtype=np.float32) * dt(sigma)
    P[n - n_out:] = g.uniform(-1.2, 1.2, (n_out, dim))
    return P[g.permutation(n)]


def _batch(case, seed):
    """Uneven clouds as synth.batched_clouds draws them (spirals, helices, segment chains, noise a
    fraction of the extent, radius four times the noise)."""
    m = case["clouds"]
    clouds = synth.batched_clouds(count=m, seed=seed, min_pts=case["lo"], max_pts=case["hi"], dtype=_dtype(case))
    return [(p[:, :case["dim"]], a, b) for p, a, b in clouds]


def _capacity(case):
    return min(case.get("n", 1 << 19), 1 << 19)


def prepare(case, seed):
    dt = _dtype(case)
    kind = case["kind"]
    st = dict(case=case, ctx=Context(case["dim"], dt), used=0)
    c = st["ctx"]
    # the caller's result buffer: how many points there will be follows from the data, so it
    # has room for as many as there can be (or a generous limit), zeros after the last one
    st["out"] = np.zeros((_capacity(case), case["dim"]), dtype=dt)
    if kind == "batch":
        st["clouds"] = _batch(case, seed)
        return st
    P = _cloud(case, seed)
    c.set_points(P)
    if kind in ("evolve", "iteration", "decimate"):
        st["S0"], _ = c.choose(case["r"])
    if kind == "vjp":
        S0, _ = c.choose(case["r"])
        g = torch.from_numpy(_upstream(case, seed, len(S0))).cuda()
        st["gS"] = g
        st["gP"] = torch.empty((case["dim"], case["n"]), dtype=g.dtype, device="cuda")
        st["gS0"] = torch.zeros(case["dim"] * _capacity(case), dtype=g.dtype, device="cuda")
        torch.cuda.synchronize()
    return st


def _upstream(case, seed, K):
    """dL/dS_T as a caller's loss gives it, one column per chosen point."""
    g = np.random.Generator(np.random.PCG64(seed + 77))
    return np.ascontiguousarray(g.normal(0.0, 1.0, (case["dim"], K)).astype(_dtype(case)))


# ---------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------
def _put(st, points, first=0):
    """points as rows `first`.. of the result buffer; returns the row after them."""
    end = first + len(points)
    st["out"][first:end, :points.shape[1]] = points
    return end


def _whole(st, end):
    """The result buffer and its number of points; rows a larger earlier result used are cleared."""
    if st["used"] > end:
        st["out"][end:st["used"]] = 0
    st["used"] = end
    return {"points": st["out"], "count": end}


def _flags(st, key, values):
    buf = st.setdefault(key, np.zeros(_capacity(st["case"]), dtype=np.int32))
    buf[:len(values)] = values
    return buf


def run(st):
    case, c = st["case"], st["ctx"]
    kind = case["kind"]
    if kind == "ridge":
        return _whole(st, _put(st, c.ridge_detection(case["r"], 2 * case["r"], max_evolve_iters=case["cap"])))
    if kind == "tiled":
        return _whole(st, _put(st, c.tiled(case["algorithm"], case["r"], 2 * case["r"], case["capacity"],
                                           [case["tiles"]] * case["dim"], refinement=case["refine"],
                                           max_evolve_iters=100)))
    if kind == "batch":
        res = c.batch([p for p, _, _ in st["clouds"]], [a for _, a, _ in st["clouds"]],
                      [b for _, _, b in st["clouds"]], max_evolve_iters=case["cap"])
        end = 0
        for x in res:
            end = _put(st, x, end)
        return _whole(st, end) | {"counts": np.array([len(x) for x in res])}
    if kind == "evolve":
        c.set_chosen(st["S0"])
        c.evolve_fixed(case["r"], case["iters"])
        return _whole(st, _put(st, c.points()))
    if kind == "iteration":
        c.set_chosen(st["S0"])
        points, flag, counts, sums, labels, moved = c.evolve_iteration(case["r"])
        total = st.setdefault("sums", np.zeros_like(st["out"]))
        total[:len(sums)] = sums
        return _whole(st, _put(st, points)) | {"flag": flag, "counts": _flags(st, "counts", counts), "sums": total,
                                               "labels": labels, "moved": _flags(st, "moved", moved)}
    if kind == "choose":
        points, idx = c.choose(case["r"])
        return _whole(st, _put(st, points)) | {"indices": _flags(st, "indices", idx)}
    if kind == "decimate":
        c.set_chosen(st["S0"])
        points, keep = c.decimate(2 * case["r"], DECIMATE_NO_COPY if case["no_copy"] else DECIMATE)
        return _whole(st, _put(st, points)) | {"keep": _flags(st, "keep", keep)}
    if kind == "vjp":
        c.choose(case["r"])
        c.evolve_fwd(case["r"], case["iters"], case["every"])
        c.evolve_bwd_device(st["gS"].data_ptr(), st["gP"].data_ptr(), st["gS0"].data_ptr(), seed_to_points=True)
        return _whole(st, _put(st, c.points())) | {"grad_points": st["gP"], "grad_seeds": st["gS0"]}
    raise ValueError(kind)


def work(case):
    """Every input coordinate read once; per sample one distance to its chosen point and its add
    to that point's sum, once per iteration where the call fixes the count.  The number of
    iterations and of chosen points of a whole detection follows from its data, so neither is
    counted."""
    v = 4 if case["dtype"] == "f32" else 8
    d = case["dim"]
    n = case["n"] if "n" in case else int(case["clouds"] * (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"]))
    it = case.get("iters", 1)
    b, f = n * d * v, 4.0 * n * d * it
    if case["kind"] == "iteration":
        b += 4 * n                       # the labels
    if case["kind"] == "vjp":
        b += n * d * v                   # the gradient of every sample
        f += n * d * it
    return {"bytes": float(b), "flops": float(f)}


# ---------------------------------------------------------------------------------------
# 64-bit values
# ---------------------------------------------------------------------------------------
def _nearest(P, S, rsq):
    """Label of every sample: its nearest chosen point, or -1 beyond the radius."""
    lab = torch.empty(len(P), dtype=torch.int64, device=P.device)
    for a in range(0, len(P), 1 << 15):
        p = P[a:a + (1 << 15)]
        D = torch.zeros((len(p), len(S)), dtype=torch.float64, device=P.device)
        for d in range(P.shape[1]):
            D += (p[:, d:d + 1] - S[None, :, d]) ** 2
        m, i = D.min(dim=1)
        lab[a:a + len(p)] = torch.where(m <= rsq, i, torch.full_like(i, -1))
    return lab


def _evolve_step(P, S, rsq, eps):
    lab = _nearest(P, S, rsq)
    hit = lab >= 0
    cnt = torch.bincount(lab[hit], minlength=len(S)).to(torch.float64)
    sums = torch.zeros_like(S).index_add_(0, lab[hit], P[hit])
    mean = sums / cnt.clamp(min=1.0)[:, None]
    mv = (cnt > 0)[:, None] & ((mean - S).abs() > 2 * mean.abs() * cnt[:, None] * eps)
    return torch.where(mv, mean, S), lab, cnt, sums, mv


def _greedy(X, r, most):
    """Indices of the greedy ball cover of X in its own precision (a sample is chosen unless an
    earlier chosen one covers it): the chosen set the caller's evolve starts from.  None beyond
    `most` chosen points."""
    idx, rsq = [0], torch.tensor(r, dtype=X.dtype) ** 2
    covered = torch.zeros(len(X), dtype=torch.bool, device=X.device)
    while len(idx) <= most:
        D = torch.zeros(len(X), dtype=X.dtype, device=X.device)
        for d in range(X.shape[1]):
            D += (X[:, d] - X[idx[-1], d]) ** 2
        covered |= D <= rsq.to(X.device)
        covered[:idx[-1] + 1] = True
        nxt = int(torch.argmin(covered.to(torch.uint8)))
        if bool(covered[nxt]):
            return idx
        idx.append(nxt)
    return None


def exact(case, seed):
    """Whole detections, choose and decimate return points that thresholded decisions select: in
    64 bits another set may be selected, so they have no 64-bit value to be compared with.  The
    evolve phases do, from the same chosen points."""
    if case["kind"] not in ("evolve", "iteration", "vjp"):
        return None
    dt = _dtype(case)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    X = torch.from_numpy(_cloud(case, seed)).to(dev)
    pairs = 2e11 if dev == "cuda" else 3e9
    idx = _greedy(X, case["r"], most=min(20000, int(pairs / (len(X) * case.get("iters", 1)))))
    if idx is None:
        return None
    P = X.to(torch.float64)
    at = torch.tensor(idx, device=dev)
    S = P[at]
    rsq, eps = float(dt(case["r"])) ** 2, float(np.finfo(dt).eps)
    if case["kind"] == "iteration":
        S1, _, _, sums, _ = _evolve_step(P, S, rsq, eps)
        return {"points": _padded(case, S1), "count": None, "flag": None, "counts": None, "sums": _padded(case, sums),
                "labels": None, "moved": None}
    steps = []
    for _ in range(case["iters"]):
        S, lab, cnt, _, mv = _evolve_step(P, S, rsq, eps)
        steps.append((lab, cnt, mv))
    if case["kind"] == "evolve":
        return {"points": _padded(case, S), "count": None}
    G = torch.from_numpy(_upstream(case, seed, len(idx)).astype(np.float64).T.copy()).to(dev)
    gP = torch.zeros_like(P)
    for lab, cnt, mv in reversed(steps):
        A = torch.where(mv, G / cnt.clamp(min=1.0)[:, None], torch.zeros_like(G))
        hit = lab >= 0
        gP[hit] += A[lab[hit]]
        G = torch.where(mv, torch.zeros_like(G), G)
    gP[at] += G
    return {"points": _padded(case, S), "count": None, "grad_points": gP.T.contiguous().cpu(),
            "grad_seeds": _padded(case, G.T.reshape(-1), case["dim"])}


def _padded(case, rows, scale=1):
    out = torch.zeros((_capacity(case) * scale, *rows.shape[1:]), dtype=torch.float64)
    out[:len(rows)] = rows.cpu()
    return out
