"""The ray cast's shortcuts come out as the arithmetic they stand for (CPU).

The device decides a node's level-of-detail test from a range of voxel half
sizes (lod_range) and a node's step count from products with reciprocals
(exit_steps) wherever rounding cannot change the outcome, and takes c / 255,
quotients by the pool's sides and the trilinear weights from products.  The
functions and constants that the kernels are built from (vox_raymath.h), built
here without a device, against the stated arithmetic on drawn rays, with square
roots and reciprocals one unit in the last place off either way."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from voxvizthesis_amd import _lib
from voxvizthesis_amd.gvserve import camera, raycast_params

f = np.float32
HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def rm(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("raymath") / "raymath_check.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off",
                    "-Wall", "-Wno-unknown-pragmas", os.path.join(HERE, "cpp", "raymath_check.cpp"),
                    "-o", so], check=True)
    L = C.CDLL(so)
    L.rm_uniforms.restype = C.c_void_p
    L.rm_uniforms.argtypes = [C.POINTER(_lib.VoxCamera), C.POINTER(_lib.VoxRaycastParams), C.c_int,
                              C.c_uint32, C.c_uint32, C.c_uint32]
    for name, args in (("rm_free", [C.c_void_p]), ("rm_odd_step", [C.c_void_p]),
                       ("rm_lod", [C.c_void_p, C.c_int, C.c_void_p, C.c_int] + [C.c_void_p] * 2),
                       ("rm_exit", [C.c_void_p, C.c_int] + [C.c_void_p] * 4 + [C.c_int] +
                        [C.c_void_p] * 4),
                       ("rm_div_by", [C.c_int, C.c_void_p, C.c_float, C.c_void_p]),
                       ("rm_weigh", [C.c_int] + [C.c_void_p] * 4), ("rm_unorm8_256", [C.c_uint32])):
        getattr(L, name).argtypes = args
    L.rm_unorm8_256.restype = C.c_float
    return L


def ptr(*arrays):
    return [a.ctypes.data for a in arrays]


def uniforms(rm, pos, look, up, fov, W, H, lo, hi, levels=7, brick=16, pool=144, wide=0, step=0.0):
    U = rm.rm_uniforms(C.byref(camera(pos, look, up, fov, W, H)),
                       C.byref(raycast_params(lo, hi, ray_step=step)), levels, brick, pool, wide)
    assert U
    return U


# a camera in the volume, beside it, far off; wide and narrow pixels; a volume
# off the unit cube, and ones that are long on one axis
@pytest.mark.parametrize("spread,fov,height,shift,size", [
    (0.5, 60.0, 1080, 0.0, (1, 1, 1)), (0.05, 60.0, 1080, 0.0, (1, 1, 1)),
    (0.002, 70.0, 64, 0.0, (1, 1, 1)), (3.0, 35.0, 720, 0.0, (1, 1, 1)),
    (40.0, 20.0, 1440, 0.0, (1, 1, 1)), (0.5, 60.0, 1080, 3.25, (1, 1, 1)),
    (0.5, 60.0, 1080, -700.0, (32, 8, 2)), (0.5, 60.0, 480, 0.0, (0.01, 0.01, 4))])
def test_lod_range_never_decides_against_the_test(rm, spread, fov, height, shift, size):
    rng = np.random.default_rng(int(1000 * spread) + height)
    n, levels, decided, total = 4000, 10, 0, 0
    size = np.array(size, np.float64)
    for _ in range(12):
        look = rng.normal(size=3)
        look /= np.linalg.norm(look)
        up = np.cross(look, rng.normal(size=3))
        up /= np.linalg.norm(up)
        lo = np.full(3, shift)
        pos = lo + size * (0.5 + spread * rng.normal(size=3))
        U = uniforms(rm, pos, look, up, fov, height * 16 // 9, height, lo, lo + size)
        p = rng.random((n, 3)).astype(f)   # unit-volume coordinates
        sure, stop = np.empty((2, n, levels), np.uint8)
        for ulp in (-1, 0, 1):
            rm.rm_ulp(ulp)
            rm.rm_lod(U, n, *ptr(p), levels, *ptr(sure, stop))
            assert not (sure & stop).any()
        decided += int(sure.sum())
        total += sure.size
        rm.rm_free(U)
    print(f"decided {decided} of {total}")
    assert spread > 1 or max(size) / min(size) > 4 or decided > 0.2 * total


@pytest.mark.parametrize("levels", [2, 5, 8])
def test_exit_steps_equal_the_divided_ones(rm, levels):
    rng = np.random.default_rng(levels)
    n = 200000
    U = uniforms(rm, (0.5, -1.0, 0.5), (0, 1, 0), (0, 0, 1), 60.0, 64, 64, (0,) * 3, (1,) * 3,
                 levels)
    step = 0.5 / (16 << (levels - 1))
    d = rng.normal(size=(n, 3))
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(f)
    d[rng.random((n, 3)) < 0.02] = 0
    d[rng.random((n, 3)) < 0.01] *= f(1e-40)             # reciprocals that overflow
    size = rng.choice([1.0, 0.125, 2.0 ** -6], (n, 1))
    mn = (np.floor(rng.random((n, 3)) / size) * size).astype(f)
    mx = (mn + size).astype(f)
    p = (mn + size * rng.random((n, 3))).astype(f)
    p = np.where(rng.random((n, 3)) < 0.02, mn, p)       # on a face, and just outside
    p[: n // 50] = np.nextafter(mx[: n // 50], f(2))
    # quotients at and near whole numbers: k steps before the exit face in x
    k = rng.integers(1, 60, n // 4)[:, None] * step
    m = slice(n - n // 4, n)
    p[m] = np.where(d[m] > 0, mx[m] - d[m] * k, mn[m] - d[m] * k).astype(f)
    for e in (0, 1, levels - 1):
        for ulp in (-1, 0, 1):
            rm.rm_ulp(ulp)
            fast, want, used = np.empty((3, n), np.int32)
            sure = np.empty(n, np.uint8)
            rm.rm_exit(U, n, *ptr(p, d, mn, mx), e, *ptr(fast, sure, want, used))
            assert (used == want).all() and (fast == want)[sure != 0].all()
            assert sure[: n // 2].mean() > 0.7
    rm.rm_free(U)


def test_unorm8_is_the_rounded_quotient(rm):
    for c in range(256):
        assert f(rm.rm_unorm8_256(c)) == f(256) * (f(c) / f(255))


# brick texels per axis of wide pools (B + 2) and of texture pools
@pytest.mark.parametrize("b", [3, 6, 9, 18, 34, 66, 100, 144, 288, 720, 1023, 1024])
def test_div_by_is_the_rounded_quotient(rm, b):
    rng = np.random.default_rng(b)
    a = np.concatenate([rng.random(40000) * 16, np.exp2(rng.uniform(-149, 10, 40000)),
                        np.arange(1024), [0.0]]).astype(f)
    out = np.empty_like(a)
    rm.rm_div_by(a.size, *ptr(a), b, *ptr(out))
    assert np.array_equal(out, a / f(b))


def test_weighed_samples_equal_the_products(rm):
    rng = np.random.default_rng(1)
    n = 20000
    t = rng.integers(0, 2 ** 32, (n, 8), dtype=np.uint32) * (rng.random((n, 8)) < 0.7)
    t = np.ascontiguousarray(t, np.uint32)
    w = rng.integers(0, 257, (n, 3)).astype(f)
    got, want = np.empty((2, n, 4), f)
    rm.rm_weigh(n, *ptr(t, w, got, want))
    assert np.array_equal(got, want)


def test_brick_steps_that_are_no_number_are_found(rm):
    tiny = float(np.finfo(f).smallest_subnormal)
    view = ((0.5, -1.0, 0.5), (0, 1, 0), (0, 0, 1), 60.0, 65, 65)
    for lo, hi, step, odd in [((0,) * 3, (1,) * 3, 0.0, 0), ((0,) * 3, (2 * tiny, 1, 1), 0.0, 1),
                              ((0,) * 3, (1, 1e38, 1), 0.45, 1), ((0,) * 3, (1, 1e-30, 1), 0.0, 0)]:
        for wide in (0, 1):
            U = uniforms(rm, *view, lo, hi, levels=4, brick=8, pool=100, wide=wide, step=step)
            assert rm.rm_odd_step(U) == odd
            rm.rm_free(U)
