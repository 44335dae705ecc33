"""CPU check of the rounding bound behind the neighbour search's sweep on halves.

Points are kept relative to the frame of their tile, one half per coordinate, times a power of two; a candidate's
distance is |q - c|^2 + beta_f(x) - 2 q'.x' with f the query's frame and c the candidate's, less a bound, and a
candidate that the sweep drops is proven farther than the neighbours by that being a LOWER bound of the distance.  Here
the arithmetic is restated in numpy (halves, sums in fp32) and compared with distances in 64 bits, with frames the
points lie close to and far from, near and far from the origin, and with coordinates that underflow as halves."""
import numpy as np
import pytest


def halves(v, scale):
    w = (v * np.float32(scale)).astype(np.float32)
    w[np.abs(w) < np.float32(2.0 ** -14)] = 0.0
    return w.astype(np.float16)


def lower_bounds(q, x, f, c, reach):
    """The sweep's keys for queries q of frame f against candidates x (one tile) of frame c."""
    d = q.shape[1]
    scale = 2.0 ** (13 - int(np.floor(np.log2(reach))))
    s2 = np.float32(0.5 * scale * scale)
    qr, xr = (q - f).astype(np.float32), (x - c).astype(np.float32)
    qh, xh = halves(qr, scale), halves(xr, scale)

    def lengths(v, h):
        lost = v - h.astype(np.float32) / np.float32(scale)
        return [(np.sqrt((e.astype(np.float32) ** 2).sum(1, dtype=np.float32)) * np.float32(1.001)) for e in (v, lost)]

    q_len, q_eps = lengths(qr, qh)
    x_len, x_eps = (v.max() for v in lengths(xr, xh))
    beta = ((xr * xr).sum(1, dtype=np.float32) - np.float32(2) * (xr * (f - c)).sum(1, dtype=np.float32)).astype(np.float32)
    d2 = ((f - c) ** 2).sum(dtype=np.float32)
    beta_q = ((qr * qr).sum(1, dtype=np.float32) - np.float32(2) * (qr * (c - f)).sum(1, dtype=np.float32)).astype(np.float32)
    kap = np.float32(5 * (d + 8) * 2.0 ** -24)
    frame_len = np.sqrt(d2) * np.float32(1.001)
    off = beta_q + d2 - np.float32(0.25) * kap * (q_len + frame_len) ** 2
    split = q_len * x_eps + q_eps * (x_len + x_eps)
    off = off - (np.float32(2.02) * split + kap * x_len * (2 * q_len + x_len + 2 * frame_len))
    # Products accumulated in fp32 one after the other from -beta / 2 (the matrix unit's order is another one).
    acc = np.repeat((-beta * s2)[None], len(q), 0).astype(np.float32)
    for k in range(d):
        acc = (acc + qh[:, k:k + 1].astype(np.float32) * xh[None, :, k].astype(np.float32)).astype(np.float32)
    return np.maximum(off[:, None] - acc / s2, 0.0)


@pytest.mark.parametrize("d", [5, 16, 50, 128, 784])
@pytest.mark.parametrize("kind", ["same frame", "near frames", "far frames", "far from the origin", "one far point"])
def test_keys_are_lower_bounds(d, kind):
    rng = np.random.default_rng(d)
    base = 300.0 if kind == "far from the origin" else 0.0
    f = (rng.standard_normal(d) + base).astype(np.float32)
    c = f.copy()
    if kind in ("near frames", "far from the origin"):
        c = (f + rng.standard_normal(d)).astype(np.float32)
    elif kind == "far frames":
        c = (f + 30.0 * rng.standard_normal(d)).astype(np.float32)
    q = (f + rng.standard_normal((64, d))).astype(np.float32)
    x = (c + rng.standard_normal((128, d))).astype(np.float32)
    if kind == "one far point":
        x[5] += 1e4
    reach = max(np.sqrt(((q - f) ** 2).sum(1).max()), np.sqrt(((x - c) ** 2).sum(1).max())) * 1.01
    if kind == "one far point":
        reach *= 2.0 ** 12  # (of some other tile: these points' coordinates lose bits and vanish)
    lb = lower_bounds(q, x, f, c, float(reach))
    exact = ((q.astype(np.float64)[:, None] - x.astype(np.float64)[None]) ** 2).sum(2)
    assert (lb <= exact * (1.0 + (d + 4) * 2.0 ** -24)).all()
    if kind in ("same frame", "near frames"):  # ... and near enough to tell neighbours apart
        assert (exact - lb).max() < 0.02 * exact.mean()
