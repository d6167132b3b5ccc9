"""The closed-form z-intervals of field pass 1 (fast_interval) against the float predicate they stand
for, restated in numpy float32: wherever the rule decides, its interval is the predicate's, and the
row range (ymargin) holds every row whose exact test passes.  The hardware root is within an ulp of
the correctly rounded one; the restatement moves it by one ulp either way at random."""
import numpy as np
import pytest

F = np.float32


def _root(x, rng):
    r = np.sqrt(np.maximum(x, F(0))).astype(F)
    step = rng.integers(-1, 2, r.shape)
    return np.where(step > 0, np.nextafter(r, F(np.inf)), np.where(step < 0, np.nextafter(r, F(0)), r)).astype(F)


def _sample(dx, offset, seed, n=4000, g=300):
    rng = np.random.default_rng(seed)
    dx, probe = F(dx), F(1.4)
    inv = F(1) / dx
    o = F(offset) - F(0.37)
    rad = rng.choice(np.array([1.2, 1.52, 1.55, 1.7, 1.8, 5.0], F), n)
    T = (rad + probe) if seed % 2 else np.maximum(rad - dx, F(0.05))
    T = T.astype(F)
    ss = (T * T).astype(F)  # stands for the threshold: any float will do
    az = (o + rng.uniform(3, float(dx) * g - 3, n).astype(F)).astype(F)
    # the sum S below ss, many near it and many that put an end close to a grid point
    S = (ss * rng.uniform(0, 1, n).astype(F)).astype(F)
    near = rng.random(n) < 0.3
    k = rng.integers(0, g, n).astype(F)
    e = (az - (o + k * dx)).astype(F)
    S = np.where(near & (e * e < ss), ss - e * e, S).astype(F)
    S = np.where(rng.random(n) < 0.1, ss * F(1 - 1e-4), S).astype(F)
    return rng, dx, inv, o, ss, az, S, g, rad, probe


@pytest.mark.parametrize("dx", [0.05, 0.2, 0.3, 0.5, 1.0])
@pytest.mark.parametrize("offset", [0.0, -66.0, 300.0, 20000.0])
@pytest.mark.parametrize("seed", [1, 2])
def test_decided_intervals_are_the_predicates(dx, offset, seed):
    rng, dx, inv, o, ss, az, S, g, _, _ = _sample(dx, offset, seed)
    z = np.arange(g, dtype=F)
    pz = (o + (z * dx).astype(F)).astype(F)
    e = (az[:, None] - pz[None, :]).astype(F)
    pred = (S[:, None] + (e * e).astype(F)).astype(F) < ss[:, None]
    eps = F(1.2e-7) * inv * (abs(o) + F(6) * F(g) * dx + F(4)) + F(9.6e-7) * inv * ss
    h2 = (ss - S).astype(F)
    h = (_root(h2, rng) * inv).astype(F)
    zc = ((az - o).astype(F) * inv).astype(F)
    lo, hi = (zc - h).astype(F), (zc + h).astype(F)
    d = np.minimum(np.abs(lo - np.rint(lo)), np.abs(hi - np.rint(hi)))
    sure = (d > eps) & (h2 > F(0.015625))
    L = np.maximum(np.ceil(lo).astype(int), 0)
    R = np.minimum(np.floor(hi).astype(int), g - 1)
    inside = (np.arange(g)[None, :] >= L[:, None]) & (np.arange(g)[None, :] <= R[:, None])
    assert np.array_equal(pred[sure], inside[sure])
    if abs(offset) < 1000 and dx >= 0.2:
        assert sure.mean() > 0.5  # (the sample is full of ends on grid points)


@pytest.mark.parametrize("dx", [0.05, 0.2, 0.5, 1.0])
@pytest.mark.parametrize("offset", [0.0, 300.0, 20000.0])
def test_row_range_holds_every_reached_row(dx, offset):
    rng, dx, inv, o, ss, ay, X, g, rad, probe = _sample(dx, offset, 3)
    y = np.arange(g, dtype=F)
    e = (ay[:, None] - (o + (y * dx).astype(F)).astype(F)[None, :]).astype(F)
    reached = (X[:, None] + (e * e).astype(F)).astype(F) < ss[:, None]
    h = (_root((ss - X).astype(F), rng) * inv).astype(F)
    yc = ((ay - o).astype(F) * inv).astype(F)
    ym = F(1.2e-7) * inv * (abs(o) + F(6) * F(g) * dx + F(4)) + F(1e-3) + F(6e-4) * inv * (rad + probe)
    rows = np.arange(g)[None, :]
    taken = (rows >= np.ceil(yc - h - ym)[:, None]) & (rows <= np.floor(yc + h + ym)[:, None])
    assert not (reached & ~taken).any()
