// vox_raymath.h -- the ray cast's arithmetic that needs no device memory: a frame's
// uniforms (host) and the decisions and products of the cast (host and device,
// so that a program without a device can compare its shortcuts with the
// arithmetic they stand for).  Approximate square roots and reciprocals come
// from a policy: rcp, rsqrt, sqrt, each within one unit in the last place.
#ifndef VOX_RAYMATH_H
#define VOX_RAYMATH_H

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>

#include "../../include/voxmi_serve.h"

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define VOX_HD __host__ __device__ __forceinline__
#else
#define VOX_HD inline
#endif

namespace voxmi {

constexpr int kMaxUsage = 12;  // 3 lists x 4 components per pixel

struct RayUniforms {
    float camPos[3], camUp[3], camLeft[3];
    float volMin[3], volMax[3], volScale[3];
    float look[3], right[3], upv[3];  // world ray basis: look, right*tanX, up*tanY
    float rayStep, rootVoxelHalf, pixelSize, lodScalar;
    float brickStep[3], brickDim[3], poolDim[3];
    int32_t depthMinusOne, maxPush, W, H, maxTraversals;
    int32_t rx0, ry0, rx1, ry1;  // pixels cast: [rx0, rx1) x [ry0, ry1)
    uint32_t ndim[3], pdim[3];
    // wide brick pool: word 1 of a resident node is its slot, and each brick
    // is sampled in its own (B+2)^3 texel frame (poolDim / pdim are then the
    // brick's texels per axis)
    uint32_t wide, wideSlots;
    float firstTexel[3];     // 1 / poolDim: a wide pool's first interior texel
    // brickStep is no number, or so large that a sum of it is none: the
    // kernels' instance for that casts the frame (looked at by the host)
    uint32_t oddStep;
    float invRayStep;        // about 1 / rayStep
    // Bounds of the level-of-detail test's outcome (lod_range): u about
    // camLeft - camUp, lodU at least its length, and the constants of the
    // lowest voxel size that surely spans a pixel.
    float lodVec[3], lodU, lodK1, lodK2;
};

struct v3 {
    float x, y, z;
};
VOX_HD v3 mk(float x, float y, float z) { return {x, y, z}; }
VOX_HD v3 add(v3 a, v3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
VOX_HD v3 sub(v3 a, v3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
VOX_HD v3 mul(v3 a, v3 b) { return {a.x * b.x, a.y * b.y, a.z * b.z}; }
VOX_HD v3 divv(v3 a, v3 b) { return {a.x / b.x, a.y / b.y, a.z / b.z}; }
VOX_HD v3 muls(v3 a, float s) { return {a.x * s, a.y * s, a.z * s}; }
VOX_HD float dot(v3 a, v3 b) { return (a.x * b.x + a.y * b.y) + a.z * b.z; }
VOX_HD v3 normalize(v3 v) { return muls(v, 1.0f / sqrtf(dot(v, v))); }
VOX_HD float signf(float x) { return x > 0.0f ? 1.0f : (x < 0.0f ? -1.0f : 0.0f); }
VOX_HD v3 ld3(const float* p) { return {p[0], p[1], p[2]}; }

VOX_HD float inside_count(v3 p, v3 mn, v3 mx) {
    const v3 t1 = mk(signf(p.x - mn.x), signf(p.y - mn.y), signf(p.z - mn.z));
    const v3 t2 = mk(signf(mx.x - p.x), signf(mx.y - p.y), signf(mx.z - p.z));
    return dot(t1, t2);
}

// x^(2^n) by squaring.
VOX_HD float pow2n(float x, int n) {
    for (int i = 0; i < n; ++i) x = x * x;
    return x;
}

// ComputeMinRayBoxIntersection (GigaVoxels.frag 155-180): the smallest
// positive-direction exit time over the six faces, 4 if none.  (A ray leaves
// an axis through the face its direction points at: mx for d > 0, mn for
// d < 0.)
VOX_HD float exit_time(v3 p, v3 d, v3 mn, v3 mx) {
    float tMin = 4.0f;
    const float dc[3] = {d.x, d.y, d.z};
    const float x[3] = {d.x > 0.0f ? mx.x - p.x : p.x - mn.x, d.y > 0.0f ? mx.y - p.y : p.y - mn.y,
                        d.z > 0.0f ? mx.z - p.z : p.z - mn.z};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        // -x * (-1 / d) and x / |d| round alike
        const float t = x[a] / fabsf(dc[a]);
        if (dc[a] != 0.0f && t < tMin && fabsf(t) > 0.0f) tMin = t;
    }
    return tMin;
}

// Steps of 2^n ray steps to the exit of a node's box: (int)(exit_time / step)
// + 1.  First from products with reciprocals: times and quotient are then
// within 16 unit roundoffs of the divided ones, so where the quotient less
// and plus a millionth of itself truncate to one integer, that integer is
// the divided quotient's too; else (a few rays in a thousand) it is divided
// out.  rd: 1 / |d| per axis, 0 for d = 0.
template <class Approx>
VOX_HD v3 rcp_dir(v3 d) {
    return {d.x != 0.0f ? Approx::rcp(fabsf(d.x)) : 0.0f,
            d.y != 0.0f ? Approx::rcp(fabsf(d.y)) : 0.0f,
            d.z != 0.0f ? Approx::rcp(fabsf(d.z)) : 0.0f};
}
VOX_HD bool exit_steps_sure(const RayUniforms& U, v3 p, v3 d, v3 rd, v3 mn, v3 mx, int n,
                            int& steps) {
    const float x = d.x > 0.0f ? mx.x - p.x : p.x - mn.x;
    const float y = d.y > 0.0f ? mx.y - p.y : p.y - mn.y;
    const float z = d.z > 0.0f ? mx.z - p.z : p.z - mn.z;
    const float tx = x * rd.x, ty = y * rd.y, tz = z * rd.z;
    // a time of zero (a point on its exit face, or d = 0) does not count
    float t = 4.0f;
    t = tx != 0.0f ? fminf(t, tx) : t;
    t = ty != 0.0f ? fminf(t, ty) : t;
    t = tz != 0.0f ? fminf(t, tz) : t;
    const float q = ldexpf(t * U.invRayStep, -n);
    const float e = fabsf(q) * 1.0e-6f;
    steps = (int)(q - e) + 1;
    // (a ray of a direction so flat that its reciprocal overflows fails the
    // comparison, as does a quotient beyond an integer's reach)
    return (int)(q - e) == (int)(q + e) && fabsf(q) < 1.0e6f &&
           fmaxf(rd.x, fmaxf(rd.y, rd.z)) < 1.0e30f;
}
VOX_HD int exit_steps(const RayUniforms& U, v3 p, v3 d, v3 rd, v3 mn, v3 mx, int n) {
    int steps;
    if (exit_steps_sure(U, p, d, rd, mn, mx, n, steps)) return steps;
    return (int)(exit_time(p, d, mn, mx) / (U.rayStep * ldexpf(1.0f, n))) + 1;
}

// ComputeVoxelSize (GigaVoxels.frag 483-490) * LodScalar: whether a voxel of half
// size h at p is below a pixel.
VOX_HD bool lod_stops(const RayUniforms& U, v3 p, v3 cam, float h) {
    const v3 up = muls(ld3(U.camUp), h), left = muls(ld3(U.camLeft), h);
    const v3 ll = normalize(sub(add(sub(p, up), left), cam));
    const v3 ur = normalize(sub(sub(add(p, up), left), cam));
    const float proj = (1.0f - dot(ll, ur)) * U.lodScalar;
    return U.pixelSize > proj;
}

// The level-of-detail test (GigaVoxels.frag 483-490: a node is too small
// when 1 - dot(normalize(ll), normalize(ur)), ll and ur the rays to two
// corners d +- h u of its voxel of half size h, times LodScalar is below
// PixelSize) mostly comes out the same way whatever its rounding.  Its angle
// has sin >= s = 2 h |d x u| / (|d|^2 + h^2 |u|^2).  The computed corners are
// off by at most e = 7 M unit roundoffs (M: the largest coordinates that
// meet, on the host), which turns each ray by at most (pi / 2) e / m, m >=
// |d| / 2 the shorter of the two; and the computed dot is at most 12 unit
// roundoffs (here: 16) above the cosine.  With 1 - cos t >= 0.459 t^2 for
// t <= 1, the test surely goes on where
//   h |u| <= |d| / 2   and   1.6 h |d x u| >= |d|^2 K1 + |d| K2,
// K1 = sqrt(2.18 (PixelSize / LodScalar + 2^-20)), K2 = 2 pi e: a range of
// h, found once per ray position for all the levels down from the root.
// Outside it (far away, or a camera within two root voxels) the test is
// computed as it stands.  With the loops of cast_pixel and the samples' loads
// and weights as they are here, a 1080p frame of the 1024^3 tree went from
// 2.60 to 0.91 ms: the test's two normalisations a level were near half of
// its instructions.
template <class Approx>
VOX_HD void lod_range(const RayUniforms& U, v3 p, v3 cam, float& hLo, float& hHi) {
    const v3 d = sub(p, cam), u = ld3(U.lodVec);
    const v3 c = mk(d.y * u.z - d.z * u.y, d.z * u.x - d.x * u.z, d.x * u.y - d.y * u.x);
    const float A = dot(d, d), C2 = dot(c, c);
    hLo = INFINITY;
    hHi = 0.0f;
    // (a ray along u, where the cross product cancels, has no range)
    if (C2 >= 1.0e-6f * A * U.lodU * U.lodU) {
        const float rA = Approx::sqrt(A);
        hLo = (A * U.lodK1 + rA * U.lodK2) * Approx::rsqrt(C2);
        hHi = rA * 0.49f * Approx::rcp(U.lodU);
    }
}

// 256 (c / 255) for a channel c = 0 .. 255, c / 255 the correctly rounded
// quotient: one fused product (all 256 compared with the division; the scale
// changes no rounding).
VOX_HD float unorm8_256(uint32_t c) {
    const float f = (float)c;
    return __builtin_fmaf(f, 0x1.010102p-8f, f);
}

// a / b for a whole b below 2^23 whose rounded reciprocal r is at hand: the
// product a r is within one unit in the last place of the quotient, and one
// fused remainder step then rounds it correctly (Markstein 1990; b's
// significand is not all ones).  A numerator so small that the remainder
// would be subnormal is divided out.
VOX_HD float div_by(float a, float b, float r) {
    if (fabsf(a) < 0x1p-80f && a != 0.0f) return a / b;
    const float q = a * r;
    return __builtin_fmaf(__builtin_fmaf(-q, b, a), r, q);
}
VOX_HD v3 div_pool(const RayUniforms& U, v3 a) {
    return {div_by(a.x, U.poolDim[0], U.firstTexel[0]), div_by(a.y, U.poolDim[1], U.firstTexel[1]),
            div_by(a.z, U.poolDim[2], U.firstTexel[2])};
}

// The products of three weights are whole 2^24ths (at most 24 bits) and so
// exact in any order; the channels' scale of 256 is taken out with theirs.
VOX_HD void weigh_sample(const uint32_t (&t)[8], const float (&w)[3],
                                             float r[4]) {
    const float z[2] = {(256.0f - w[2]) * 0x1p-32f, w[2] * 0x1p-32f};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float wx = (k & 1) ? w[0] : 256.0f - w[0];
        const float wy = ((k >> 1) & 1) ? w[1] : 256.0f - w[1];
        const float wk = (wx * wy) * z[k >> 2];
        const uint32_t v = t[k];
        const float c[4] = {wk * unorm8_256(v & 255u), wk * unorm8_256((v >> 8) & 255u),
                            wk * unorm8_256((v >> 16) & 255u), wk * unorm8_256(v >> 24)};
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = k == 0 ? c[i] : r[i] + c[i];
    }
}

// Uniforms of one frame (GigaVoxelsRenderer.cpp 1650-1816), in float like
// the renderer's QVector3D arithmetic.
inline bool ray_uniforms(const vox_camera& cam, const vox_raycast_params& prm, int levels,
                  const uint32_t B[3], const uint32_t poolDims[3], uint32_t poolWide,
                  const uint32_t ndim[3], RayUniforms& U) {
    std::memset(&U, 0, sizeof(U));
    float T[3], S[3];
    for (int a = 0; a < 3; ++a) {
        T[a] = (prm.vol_min[a] + prm.vol_max[a]) * 0.5f;
        S[a] = prm.vol_max[a] - prm.vol_min[a];
        if (!(S[a] > 0.0f)) return false;
        U.volScale[a] = S[a];
        U.volMin[a] = (prm.vol_min[a] - T[a]) / S[a] + 0.5f;
        U.volMax[a] = (prm.vol_max[a] - T[a]) / S[a] + 0.5f;
        U.camPos[a] = (cam.position[a] - T[a]) / S[a] + 0.5f;
        U.camUp[a] = cam.up[a];
    }
    // left = up x look
    U.camLeft[0] = cam.up[1] * cam.look[2] - cam.up[2] * cam.look[1];
    U.camLeft[1] = cam.up[2] * cam.look[0] - cam.up[0] * cam.look[2];
    U.camLeft[2] = cam.up[0] * cam.look[1] - cam.up[1] * cam.look[0];
    const float tanY = std::tan(cam.fov_y_deg * 0.5f * 3.14159265358979f / 180.0f);
    const float tanX = tanY * (float)cam.width / (float)cam.height;
    for (int a = 0; a < 3; ++a) {
        U.look[a] = cam.look[a];
        U.right[a] = -U.camLeft[a] * tanX;
        U.upv[a] = cam.up[a] * tanY;
    }
    // RayStepSize: half the smallest voxel edge of the unit volume
    const uint32_t Nmax = std::max(B[0], std::max(B[1], B[2])) << (levels - 1);
    U.rayStep = prm.ray_step > 0.0f ? prm.ray_step : (1.0f / (float)Nmax) * 0.5f;
    if (!(U.rayStep >= 1.0e-5f)) return false;  // bounds the samples per node
    U.lodScalar = prm.lod_scalar > 0.0f ? prm.lod_scalar : 10.0f;
    // BrickStepVector = (1 / pool) * (rayStep * 2^(L-1) * S) / (S / B)
    const float pow2 = std::ldexp(1.0f, levels - 1);
    for (int a = 0; a < 3; ++a) {
        const float rayStepRoot = (S[a] * U.rayStep) * pow2;
        const float rootVoxel = S[a] / (float)B[a];
        const float ratio = rayStepRoot / rootVoxel;
        // a wide pool is sampled one brick at a time: its texels are the frame
        const uint32_t pd = poolWide ? B[a] + 2u : poolDims[a];
        U.brickStep[a] = (1.0f / (float)pd) * ratio;
        // (the edge of a box below the smallest floats: 0 / 0)
        if (!(std::fabs(U.brickStep[a]) < 1.0e30f)) U.oddStep = 1u;
        U.brickDim[a] = (float)B[a];
        U.poolDim[a] = (float)pd;
        U.pdim[a] = pd;
        U.ndim[a] = ndim[a];
    }
    U.wide = poolWide;
    U.wideSlots = poolWide ? poolDims[2] / (B[2] + 2u) : 0u;
    for (int a = 0; a < 3; ++a) U.firstTexel[a] = 1.0f / U.poolDim[a];
    U.invRayStep = 1.0f / U.rayStep;
    const float bx = (float)B[0], by = (float)B[1], bz = (float)B[2];
    const float minB = bx < ((by < bz) ? by : bz) ? bx : bz;  // renderer's ternary
    U.rootVoxelHalf = (1.0f / minB) * 0.5f;
    // PixelSize: 1 - cos of the angle between the rays through the centre
    // pixel corner and its diagonal neighbour (Camera::getPixelSize).
    {
        const double W = cam.width, H = cam.height;
        double r0[3], r1[3];
        for (int a = 0; a < 3; ++a) {
            const double sx0 = 2.0 * (W * 0.5) / W - 1.0, sy0 = 2.0 * (H * 0.5) / H - 1.0;
            const double sx1 = 2.0 * (W * 0.5 + 1.0) / W - 1.0, sy1 = 2.0 * (H * 0.5 + 1.0) / H - 1.0;
            r0[a] = cam.look[a] + (double)U.right[a] * sx0 + (double)U.upv[a] * sy0;
            r1[a] = cam.look[a] + (double)U.right[a] * sx1 + (double)U.upv[a] * sy1;
        }
        const double n0 = std::sqrt(r0[0] * r0[0] + r0[1] * r0[1] + r0[2] * r0[2]);
        const double n1 = std::sqrt(r1[0] * r1[0] + r1[1] * r1[1] + r1[2] * r1[2]);
        const double c = (r0[0] * r1[0] + r0[1] * r1[1] + r0[2] * r1[2]) / (n0 * n1);
        U.pixelSize = (float)(1.0 - c);
    }
    // the constants of lod_range, each 3 % or more on the safe side
    {
        double up = 0.0, left = 0.0, M = 0.0, mUp = 0.0, mLeft = 0.0;
        for (int a = 0; a < 3; ++a) {
            U.lodVec[a] = U.camLeft[a] - U.camUp[a];
            up += (double)U.camUp[a] * U.camUp[a];
            left += (double)U.camLeft[a] * U.camLeft[a];
            M = std::max({M, std::fabs((double)U.volMin[a]) + std::fabs((double)U.camPos[a]),
                          std::fabs((double)U.volMax[a]) + std::fabs((double)U.camPos[a])});
            mUp = std::max(mUp, std::fabs((double)U.camUp[a]));
            mLeft = std::max(mLeft, std::fabs((double)U.camLeft[a]));
        }
        M += 2.0 * U.rootVoxelHalf * (mUp + mLeft);
        const double tau =
            std::max(0.0, (double)U.pixelSize / U.lodScalar) * (1.0 + 1e-5) + std::ldexp(1.0, -20);
        U.lodU = (float)(1.001 * (std::sqrt(up) + std::sqrt(left)));
        U.lodK1 = (float)(1.03 * std::sqrt(2.18 * tau) / 1.6);
        U.lodK2 = (float)(1.03 * 2.0 * 3.14159265358979 * 7.0 * M * std::ldexp(1.0, -24) / 1.6);
    }
    U.depthMinusOne = levels - 1;
    U.maxPush = kMaxUsage * (int)((cam.frame % 2) + 1);
    U.W = cam.width;
    U.H = cam.height;
    const int32_t* r = prm.rect;
    if (r[0] == 0 && r[1] == 0 && r[2] == 0 && r[3] == 0) {
        U.rx0 = U.ry0 = 0;
        U.rx1 = cam.width;
        U.ry1 = cam.height;
    } else {
        if (r[0] < 0 || r[1] < 0 || r[2] > cam.width || r[3] > cam.height || r[2] <= r[0] ||
            r[3] <= r[1])
            return false;
        U.rx0 = r[0];
        U.ry0 = r[1];
        U.rx1 = r[2];
        U.ry1 = r[3];
    }
    U.maxTraversals = prm.max_traversals ? (int32_t)prm.max_traversals : 4096;
    return true;
}

}  // namespace voxmi

#endif
