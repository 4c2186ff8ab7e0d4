"""The ray cast's shortcuts come out as the arithmetic they stand for (CPU).

The device decides a node's level-of-detail test from a range of voxel half
sizes (lod_range) and a node's step count from products with reciprocals
(exit_steps) wherever rounding cannot change the outcome, and takes c / 255,
quotients by the pool's sides and the trilinear weights from products.  Restated here in fp32 and compared with the stated
arithmetic on drawn rays."""
import ctypes
import math

import numpy as np
import pytest

f = np.float32
LIBM = ctypes.CDLL("libm.so.6")
LIBM.fmaf.restype = ctypes.c_float
LIBM.fmaf.argtypes = [ctypes.c_float] * 3
U24 = 2.0 ** -24


def dot(a, b):
    return ((a[..., 0] * b[..., 0] + a[..., 1] * b[..., 1]) + a[..., 2] * b[..., 2]).astype(f)


def normalize(v):
    return (v * (f(1) / np.sqrt(dot(v, v)))[..., None]).astype(f)


def lod_constants(up, left, vol, cam, root_half, pixel, lod):
    M = max(abs(float(v)) for v in vol) + max(abs(float(c)) for c in cam)
    M += 2.0 * root_half * (np.abs(up).max() + np.abs(left).max())
    tau = max(0.0, pixel / lod) * (1 + 1e-5) + 2.0 ** -20
    return (f(1.001 * (np.linalg.norm(up) + np.linalg.norm(left))),
            f(1.03 * math.sqrt(2.18 * tau) / 1.6),
            f(1.03 * 2 * math.pi * 7 * M * U24 / 1.6))


# a camera in the volume, beside it, far off; wide and narrow pixels; a volume
# off the unit cube
@pytest.mark.parametrize("spread,fov,height,shift", [
    (0.5, 60.0, 1080, 0.0), (0.05, 60.0, 1080, 0.0), (0.002, 70.0, 64, 0.0),
    (3.0, 35.0, 720, 0.0), (40.0, 20.0, 1440, 0.0), (0.5, 60.0, 1080, 3.25)])
def test_lod_range_never_decides_against_the_test(spread, fov, height, shift):
    rng = np.random.default_rng(int(1000 * spread) + height)
    n, decided, total = 4000, 0, 0
    for _ in range(12):
        look = rng.normal(size=3)
        look /= np.linalg.norm(look)
        up = np.cross(look, rng.normal(size=3))
        up = (up / np.linalg.norm(up)).astype(f)
        look = look.astype(f)
        left = np.cross(up, look).astype(f)
        p = (rng.random((n, 3)) + shift).astype(f)
        cam = (0.5 + shift + spread * rng.normal(size=3)).astype(f)
        pixel = 1.0 - math.cos(math.sqrt(2) * 2 * math.tan(math.radians(fov) / 2) / height)
        pixel, lod = float(f(pixel)), 10.0
        root = f(1.0 / 16 * 0.5)
        lu, k1, k2 = lod_constants(up, left, (shift, 1 + shift), cam, float(root), pixel, lod)
        d = (p - cam).astype(f)
        u = (left - up).astype(f)
        c = np.stack([d[:, 1] * u[2] - d[:, 2] * u[1], d[:, 2] * u[0] - d[:, 0] * u[2],
                      d[:, 0] * u[1] - d[:, 1] * u[0]], -1).astype(f)
        A, C2 = dot(d, d), dot(c, c)
        ok = C2 >= f(1e-6) * A * lu * lu
        with np.errstate(divide="ignore", invalid="ignore"):
            # the device's square roots and reciprocals are approximate: one
            # unit in the last place, on the side that decides more
            rA = np.sqrt(A)
            lo = np.where(ok, (A * k1 + rA * k2) / np.sqrt(C2) * f(1 - 2.0 ** -21), np.inf)
            hi = np.where(ok, rA * f(0.49) / lu * f(1 + 2.0 ** -21), 0.0)
        for k in range(10):
            h = f(float(root) * 0.5 ** k)
            sure = (h >= lo) & (h <= hi)
            ll = normalize((((p - up * h) + left * h) - cam).astype(f))
            ur = normalize((((p + up * h) - left * h) - cam).astype(f))
            proj = (f(1) - dot(ll, ur)) * f(lod)
            assert not (sure & (f(pixel) > proj)).any()
            decided += int(sure.sum())
            total += n
    print(f"decided {decided} of {total}")
    assert spread > 1 or decided > 0.2 * total


@pytest.mark.parametrize("levels", [2, 5, 8])
def test_exit_steps_equal_the_divided_ones(levels):
    rng = np.random.default_rng(levels)
    n = 400000
    step = f(0.5 / (16 << (levels - 1)))
    x = np.abs(rng.random((n, 3)) * rng.choice([1.0, 0.1, 1e-3, 0.0], (n, 1))).astype(f)
    x[rng.random((n, 3)) < 0.02] = 0
    x[: n // 50] *= f(-1)                 # a point just outside the node
    # many quotients at and near whole numbers
    k = rng.integers(1, 60, n // 4)
    d = rng.normal(size=(n, 3))
    d = np.abs(d / np.linalg.norm(d, axis=1, keepdims=True)).astype(f)
    d[rng.random((n, 3)) < 0.02] = 0
    x[: n // 4] = (d[: n // 4] * (k * float(step))[:, None]).astype(f)
    with np.errstate(divide="ignore", invalid="ignore", over="ignore"):
        t = np.where((d > 0) & (x != 0), x / d, f(np.inf)).astype(f)
        want = (np.minimum(f(4), t.min(1)) / step).astype(np.float32)
        want = np.trunc(want).astype(np.int64) + 1
        for ulp in (-1, 0, 1):            # a reciprocal may be one off
            r = np.where(d != 0, (f(1) / d), f(0)).astype(f)
            r = (r * f(1 + ulp * 2.0 ** -23)).astype(f)
            tx = (x * r).astype(f)
            q = np.minimum(f(4), np.where(tx != 0, tx, f(np.inf)).min(1))
            q = (q * (f(1) / step)).astype(f)
            e = (np.abs(q) * f(1e-6)).astype(f)
            a, b = np.trunc(q - e), np.trunc(q + e)
            sure = (a == b) & (np.abs(q) < 1e6) & (r.max(1) < 1e30)
            assert (a[sure].astype(np.int64) + 1 == want[sure]).all()
            # (a quarter of the rows lie on every face: the quotient of the
            # limit 4 by the step, a whole number, which is divided out)
            assert sure[n // 4:].mean() > 0.74


def fma(a, b, c):
    """Fused multiply-add in fp32 of scalars (the C library's)."""
    return LIBM.fmaf(float(a), float(b), float(c))


def test_unorm8_is_the_rounded_quotient():
    k = float.fromhex("0x1.010102p-8")
    for c in range(256):
        assert f(fma(c, k, c)) == f(256) * (f(c) / f(255))


# brick texels per axis of wide pools (B + 2) and of texture pools
@pytest.mark.parametrize("b", [3, 6, 9, 18, 34, 66, 100, 144, 288, 720, 1023, 1024])
def test_div_by_is_the_rounded_quotient(b):
    rng = np.random.default_rng(b)
    r = f(1) / f(b)
    a = np.concatenate([rng.random(4000) * 16, np.exp2(rng.uniform(-80, 10, 4000)),
                        np.arange(1024)]).astype(f)
    for x in a:
        q = x * r
        assert f(fma(fma(-q, b, x), r, q)) == x / f(b)


def test_weight_products_are_exact():
    w = np.arange(257)
    rng = np.random.default_rng(1)
    x, y, z = (rng.choice(w, 20000) for _ in range(3))
    want = ((x / 256).astype(f) * (y / 256).astype(f)) * (z / 256).astype(f)
    got = (x.astype(f) * y.astype(f)) * (z.astype(f) * f(2.0 ** -32))
    assert (got * f(256) == want).all()
    assert (want.astype(np.float64) == x * y * z / 2.0 ** 24).all()
