"""CPU check of the rounding bound behind the neighbour search's sweep on halves (csrc/half_bound.h, compiled by itself).

Points are kept relative to the frame of their tile, one half per coordinate, times a power of two; a candidate's
distance is |q - c|^2 + beta_f(x) - 2 q'.x' with f the query's frame and c the candidate's, less a bound, and a
candidate that the sweep drops is proven farther than the neighbours by that being a LOWER bound of the distance.  Here
the arithmetic is restated in numpy (halves, sums in fp32) around the kernels' own bound and compared with distances in
64 bits, with frames the points lie close to and far from, near and far from the origin, with coordinates that
underflow as halves and with coordinates whose squares underflow."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "half_bound.h"
extern "C" float length(float sum, int D) { return tsnehip::length_bound(sum, D); }
extern "C" float offset(float len, float eps, int D, float back, float beta_q, float d2, float frame_len, float tile_eps,
                        float tile_len) {
    tsnehip::HalfQuery hq = tsnehip::half_query(len, eps, D, back);
    tsnehip::enter_frame(hq, 0, beta_q, d2, frame_len);
    return tsnehip::tile_offset(hq, tile_eps, tile_len);
}
"""


@pytest.fixture(scope="module")
def bound(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    folder = tmp_path_factory.mktemp("bound")
    (folder / "bound.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "tsne-cuda_amd", "csrc"),
                    str(folder / "bound.cpp"), "-o", str(folder / "bound.so")], check=True)
    lib = ctypes.CDLL(str(folder / "bound.so"))
    lib.length.restype = lib.offset.restype = ctypes.c_float
    f, i = ctypes.c_float, ctypes.c_int
    lib.length.argtypes, lib.offset.argtypes = [f, i], [f, f, i] + [f] * 6
    return lib


def halves(v, scale):
    w = (v * np.float32(scale)).astype(np.float32)
    w[np.abs(w) < np.float32(2.0 ** -14)] = 0.0
    return w.astype(np.float16)


def flushed(v):
    return np.where(np.abs(v) < np.float32(2.0 ** -126), np.float32(0), v)


def lower_bounds(bound, q, x, f, c, reach, flush):
    """The sweep's keys for queries q of frame f against candidates x (one tile) of frame c.  flush: what is subnormal on
    the way through the matrix unit is lost there."""
    d = q.shape[1]
    scale = 2.0 ** min(max(13 - int(np.floor(np.log2(max(reach, 1e-30)))), -60), 60)
    s2 = np.float32(0.5 * scale * scale)
    back = np.float32(-1) / s2
    qr, xr = (q - f).astype(np.float32), (x - c).astype(np.float32)
    qh, xh = halves(qr, scale), halves(xr, scale)

    def lengths(v, h):
        lost = v - h.astype(np.float32) / np.float32(scale)
        return [np.array([bound.length(s, d) for s in (e.astype(np.float32) ** 2).sum(1, dtype=np.float32)], np.float32)
                for e in (v, lost)]

    q_len, q_eps = lengths(qr, qh)
    x_len, x_eps = (v.max() for v in lengths(xr, xh))
    beta = ((xr * xr).sum(1, dtype=np.float32) - np.float32(2) * (xr * (f - c)).sum(1, dtype=np.float32)).astype(np.float32)
    d2 = ((f - c) ** 2).sum(dtype=np.float32)
    beta_q = ((qr * qr).sum(1, dtype=np.float32) - np.float32(2) * (qr * (c - f)).sum(1, dtype=np.float32)).astype(np.float32)
    frame_len = bound.length(d2, d)
    off = np.array([bound.offset(q_len[i], q_eps[i], d, back, beta_q[i], d2, frame_len, x_eps, x_len)
                    for i in range(len(q))], np.float32)
    # Products accumulated in fp32 one after the other from -beta / 2 (the matrix unit's order is another one).
    acc = np.repeat((-beta * s2)[None], len(q), 0).astype(np.float32)
    for k in range(d):
        if flush:
            acc = flushed(acc)
        acc = (acc + qh[:, k:k + 1].astype(np.float32) * xh[None, :, k].astype(np.float32)).astype(np.float32)
    return np.maximum(off[:, None] + (flushed(acc) if flush else acc) * back, 0.0)


def in_sweep_order(q, x):
    """Distances as the re-rank forms them: fp32, one dimension after the other."""
    acc = np.zeros((len(q), len(x)), np.float32)
    for k in range(q.shape[1]):
        diff = (q[:, k:k + 1] - x[None, :, k]).astype(np.float32)
        acc = (acc + diff * diff).astype(np.float32)
    return acc


def check(bound, q, x, f, c, reach, flush=False):
    d = q.shape[1]
    lb = lower_bounds(bound, q, x, f, c, float(reach), flush)
    exact = ((q.astype(np.float64)[:, None] - x.astype(np.float64)[None]) ** 2).sum(2)
    assert (lb <= exact * (1.0 + (d + 4) * 2.0 ** -24)).all()
    assert (lb <= in_sweep_order(q, x).astype(np.float64) * (1.0 + 2 * (d + 4) * 2.0 ** -24)).all()
    return lb, exact


def greatest(q, f, x, c):
    return max(np.sqrt(((q - f).astype(np.float64) ** 2).sum(1).max()), np.sqrt(((x - c).astype(np.float64) ** 2).sum(1).max()))


@pytest.mark.parametrize("d", [5, 16, 50, 128, 784])
@pytest.mark.parametrize("kind", ["same frame", "near frames", "far frames", "far from the origin", "one far point"])
def test_keys_are_lower_bounds(bound, d, kind):
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
    reach = greatest(q, f, x, c) * 1.01
    if kind == "one far point":
        reach *= 2.0 ** 12  # (of some other tile: these points' coordinates lose bits and vanish)
    lb, exact = check(bound, q, x, f, c, reach)
    if kind in ("same frame", "near frames"):  # ... and near enough to tell neighbours apart
        assert (exact - lb).max() < 0.02 * exact.mean()


@pytest.mark.parametrize("d", [5, 16, 50])
@pytest.mark.parametrize("size", [1e-12, 1e-15, 1e-17, 1e-18, 3e-19, 1e-19, 7e-20, 2e-20, 1e-21])
@pytest.mark.parametrize("flush", [False, True])
def test_keys_are_lower_bounds_where_squares_underflow(bound, d, size, flush):
    """Points that fill their tile to the same distance (the largest of the tile leaves no room to spare), frames at a
    like distance, around the origin; alone, and beside tiles that reach as far as points are let."""
    rng = np.random.default_rng(d)
    with np.errstate(under="ignore"):
        for trial in range(8):
            f = np.zeros(d, np.float32)
            c = (size * rng.standard_normal(d) * (trial % 2)).astype(np.float32)
            q = (f + size * np.sign(rng.standard_normal((64, d))) * (1.0 + 0.01 * rng.random((64, d)))).astype(np.float32)
            x = (c + size * np.sign(rng.standard_normal((128, d))) * (1.0 + 0.01 * rng.random((128, d)))).astype(np.float32)
            reach = greatest(q, f, x, c) * 1.01
            for beside in (1.0, 2.0 ** 16, 1e18 / reach):
                check(bound, q, x, f, c, reach * beside, flush)
