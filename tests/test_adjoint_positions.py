"""CPU check of how the back-projection adjoint finds its pixels
(kernels_learned.hip: k_bp_adjoint), in the kernel's arithmetic: a thread of
(angle, bin k) walks the lines of the image with tc, the position where kf = k,
in 32.32 fixed point, and takes three pixels from the first within 1/as of tc
(the integer part of tc - 1/as + 1).
  - every pixel whose weight in exact arithmetic is not a rounding error is one
    of the three, at its own weight to a few 2^-24;
  - clamped to [-3, n], the three pixels lie in the line's padding of four on
    each side, and a pixel of the image is never moved by the clamp;
  - the lines a wave leaves out hold no such pixel."""
import math

import numpy as np
import pytest

f32, f64 = np.float32, np.float64
ONE = 2.0 ** 32


def _fma(a, b, c):
    return (np.asarray(a, f64) * np.asarray(b, f64) + np.asarray(c, f64)).astype(f32)


def _geometry(ndet, th):
    c, sn, det_c = f32(math.cos(th)), f32(math.sin(th)), f32(0.5) * f32(ndet - 1)
    rows = abs(c) >= abs(sn)
    return c, sn, det_c, rows, (c if rows else -sn), (-sn if rows else c)


def positions(n, ndet, th, lines=None):
    """(first pixel before the clamp, three weights) for every (line, bin); `lines`: these only."""
    c, sn, det_c, _, slope, b = _geometry(ndet, th)
    a = f64(det_c) + (0.5 * n - 0.5) * (f64(sn) - f64(c))
    t0 = (np.arange(ndet) - a) / f64(slope)
    step = np.int64(np.rint(-f64(b) / f64(slope) * ONE))
    u = np.asarray(range(n) if lines is None else lines)[:, None]
    az = abs(slope)
    q = np.rint((t0 + (1.0 - 1.0 / f64(az))) * ONE).astype(np.int64)[None, :] + u * step
    fr = (q & 0xFFFFFFFF).astype(np.uint32).astype(f32)
    unit = az * f32(1 / ONE)
    w = [_fma(fr, -unit, az), f32(1) - abs(_fma(fr, -unit, f32(2) * az - f32(1))),
         np.maximum(_fma(fr, unit, f32(2.0 - 3.0 * f64(az))), f32(0))]
    return q >> 32, w


def _check(n, ndet, th):
    c, sn, det_c, rows, slope, b = _geometry(ndet, th)
    first, w = positions(n, ndet, th)
    assert np.abs(first).max() < 2 ** 15
    # exact kf of every (line, position), the kernel's float cos, sin and det_c
    m = 0.5 * n - 0.5
    a = f64(det_c) + m * (f64(sn) - f64(c))
    k = np.arange(ndet)[None, :]
    u = np.arange(n)[:, None]
    for off in range(-2, 5):  # the three pixels and two on each side
        t = first + off
        exact = np.maximum(0.0, 1.0 - np.abs(a + u * f64(b) + t * f64(slope) - k))
        inside = (t >= 0) & (t < n)
        got = w[off] if 0 <= off < 3 else np.zeros_like(exact)
        # position to 2^-24, its product with as, two sums and n steps of 2^-33
        assert np.abs(got - exact)[inside].max(initial=0.0) <= 8 * 2.0 ** -24 + n * 2.0 ** -33, (n, ndet, th, off)
    t = np.clip(first, -3, n)
    assert np.array_equal(np.where((first + 2 >= 0) & (first < n), first, t), t)
    moved = t != first
    assert np.all((t[moved] == -3) | (t[moved] == n))
    # the lines each wave of 64 bins walks
    dt, tc0 = f32(-f64(b) / f64(slope)), ((np.arange(ndet) - a) / f64(slope)).astype(f32)
    if abs(dt) > f32(1e-3):
        ua, ub = (f32(-2) - tc0) / dt, (f32(n) + f32(1) - tc0) / dt
        lo = np.maximum(f32(0), np.floor(np.minimum(ua, ub)) - f32(2))
        hi = np.minimum(f32(n), np.ceil(np.maximum(ua, ub)) + f32(3))
        needed = (first + 2 >= 0) & (first < n)
        assert np.all(~needed | ((u >= lo[None, :]) & (u < hi[None, :]))), (n, ndet, th)


@pytest.mark.parametrize("n", [8, 31, 64, 96, 128, 160, 512])
def test_three_pixels_hold_every_contribution(n):
    rng = np.random.default_rng(n)
    many = 48 if n < 160 else 16
    angles = [2 * math.pi * a / many for a in range(many)] + [math.pi / 4 + 1e-7, 3 * math.pi / 4 - 1e-7]
    angles += list(rng.uniform(-10, 10, 8))
    for ndet in sorted({n, int(1.4143 * n) + 1, 2 * n + 3}):
        for th in angles:
            _check(n, ndet, th)


def test_largest_geometry_stays_in_fixed_point():
    for th in (0.0, math.pi / 4, 0.7, math.pi / 2, 2.3, 3.0):
        first, _ = positions(8192, 5000, th, lines=(0, 1, 4096, 8191))
        assert np.abs(first).max() < 2 ** 15
