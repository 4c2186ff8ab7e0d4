// vox_serve.hip -- sparse-octree ray cast producing brick requests, and the
// request deduplication (C ABI in include/voxmi_serve.h).
//
// The ray cast restates VoxViz/Shaders/GigaVoxels.frag main (544-805) per
// pixel: descend from the root while the node is constant or has a resident
// brick, its projected voxel is larger than a pixel and it has children;
// at the stopping node composite its constant colour or the most recently
// descended resident brick up to the node's exit, record the node in the
// pixel's usage list, restart from the root.  fp32, no contraction, the
// shader's operation order; GLSL built-ins are defined as follows (the same
// definitions hold in the oracle):
//   normalize(v) = v * (1 / sqrt(dot(v, v))), dot = (x*x + y*y) + z*z
//   pow(x, 2^n)  = x squared n times (all exponents in the shader are 2^n)
//   texture()    = trilinear, clamp to edge, weights rounded to 8 fractional
//                  bits, unorm8 texels as c / 255
//   uvec3(v)     = truncation, negative components 0
// Rays start on the box of the octree (the rasterized front faces of the
// reference), at the camera when it is inside the box.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <new>
#include <sstream>
#include <string>
#include <vector>

#include "../../include/voxmi_serve.h"
#include "vox_internal.h"
#include "vox_raymath.h"

using namespace voxmi;

namespace {

constexpr uint32_t kConstBit = 0x40000000u;
constexpr uint32_t kResidentBit = 0x80000000u;

// The device's approximate square roots and reciprocals (vox_raymath.h).
struct HwApprox {
    static __device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
    static __device__ __forceinline__ float rsqrt(float x) { return __builtin_amdgcn_rsqf(x); }
    static __device__ __forceinline__ float sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
};

__device__ __forceinline__ void unpack_rgba(uint32_t c, float o[4]) {
    o[0] = unorm8_256(c & 255u) * 0x1p-8f;
    o[1] = unorm8_256((c >> 8) & 255u) * 0x1p-8f;
    o[2] = unorm8_256((c >> 16) & 255u) * 0x1p-8f;
    o[3] = unorm8_256(c >> 24) * 0x1p-8f;
}

// texture(BrickSampler, s): trilinear, clamp to edge.  unorm8 channel c
// reads c / 255 (no table: 32 reads a sample at addresses that differ by
// lane kept LDS busier than these few instructions do the VALU); the pool
// has at most 2^30 texels, so texel indices fit 32 bits.  The eight texels
// come as four pairs along x (x0 and x0 + 1 moved inside the edge, the pair
// then read from one side where the edge clamps it) and are loaded before
// any is used (one memory round trip per sample), then weighted in corner
// order 0..7.
// A node texture or brick pool in device memory.  Typed so, loads through
// it are global loads also where the pointer itself was read from memory (an
// octree table), which the compiler would otherwise load with flat ones.
typedef const __attribute__((address_space(1))) uint32_t* gu32;

struct pair32 {
    uint32_t a, b;
} __attribute__((packed, aligned(4)));
typedef const __attribute__((address_space(1))) pair32* gpair;

// Loads of one sample: eight texels t in corner order and the weights w,
// whole 256ths.
// Coordinates are clamped as floats (the texel numbers are whole and below
// 2^24); a pool has at most 1024 texels per axis, so indices are 24-bit
// products.  No coordinate is NaN (which reads as 0): the caller sees to that
// where RayUniforms::oddStep says that one could be (an instance of the cast
// for that: a test in the sample loop, uniform as it was, took 3.5 % of a frame).
__device__ __forceinline__ void load_sample(gu32 __restrict__ col, const RayUniforms& U, v3 s,
                                            uint32_t (&t)[8], float (&w)[3]) {
    const float c[3] = {s.x, s.y, s.z};
    float f[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float b = c[a] * U.poolDim[a] - 0.5f;
        f[a] = floorf(b);
        w[a] = rintf((b - f[a]) * 256.0f);
    }
    const float mx = U.poolDim[0] - 2.0f, my = U.poolDim[1] - 1.0f, mz = U.poolDim[2] - 1.0f;
    const bool left = f[0] < 0.0f, right = f[0] > mx;   // (a pool has B + 2 >= 3 texels per axis)
    const uint32_t x = (uint32_t)__builtin_amdgcn_fmed3f(f[0], 0.0f, mx);
    const float y0 = __builtin_amdgcn_fmed3f(f[1], 0.0f, my);
    const float z0 = __builtin_amdgcn_fmed3f(f[2], 0.0f, mz);
    const uint32_t o = __umul24(__umul24((uint32_t)z0, U.pdim[1]) + (uint32_t)y0, U.pdim[0]) + x;
    // the next row and slice where they lie inside the edge, else the same
    const uint32_t oy = f[1] >= 0.0f && f[1] < my ? U.pdim[0] : 0u;
    const uint32_t oz = f[2] >= 0.0f && f[2] < mz ? U.pdim[0] * U.pdim[1] : 0u;
    const uint32_t at[4] = {o, o + oy, o + oz, o + oy + oz};
    pair32 q[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        gpair g = (gpair)(col + at[k]);
        q[k].a = g->a;
        q[k].b = g->b;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        t[2 * k] = right ? q[k].b : q[k].a;
        t[2 * k + 1] = left ? q[k].a : q[k].b;
    }
}

__device__ __forceinline__ void blend(float dst[4], const float src[4]) {
    const float k = 1.0f - dst[3];
    dst[0] = k * src[0] + dst[0];
    dst[1] = k * src[1] + dst[1];
    dst[2] = k * src[2] + dst[2];
    dst[3] = k * src[3] + dst[3];
}

__device__ __forceinline__ uint2 fetch_node(gu32 __restrict__ tex, const RayUniforms& U,
                                            uint32_t x, uint32_t y, uint32_t z) {
    // texelFetch outside the texture reads 0 (never reached with valid pointers)
    if (x >= U.ndim[0] || y >= U.ndim[1] || z >= U.ndim[2]) return make_uint2(0u, 0u);
    // at most 1024 texels per axis: 24-bit products, 32-bit indices
    const uint32_t t = __umul24(__umul24(z, U.ndim[1]) + y, U.ndim[0]) + x;
    gpair g = (gpair)(tex + 2 * (uint64_t)t);
    return make_uint2(g->a, g->b);
}

// One pixel's ray through one octree (GigaVoxels.frag main): its FragColor
// in dst and its node usage list in usage (both start at zero here).
// Returns whether the ray met the octree's box.
template <bool kOddStep>
__device__ __forceinline__ bool cast_pixel(const RayUniforms& U, gu32 __restrict__ tex,
                                           gu32 __restrict__ pool,
                                           const float* __restrict__ jitter, int i, int j,
                                           float (&dst)[4], uint32_t (&usage)[kMaxUsage]) {
#pragma unroll
    for (int k = 0; k < kMaxUsage; ++k) usage[k] = 0u;
    dst[0] = dst[1] = dst[2] = dst[3] = 0.0f;

    // the pixel's ray, world -> unit volume
    const float sx = (2.0f * ((float)i + 0.5f)) / (float)U.W - 1.0f;
    const float sy = (2.0f * ((float)j + 0.5f)) / (float)U.H - 1.0f;
    const v3 dw = add(add(ld3(U.look), muls(ld3(U.right), sx)), muls(ld3(U.upv), sy));
    const v3 dn = divv(dw, ld3(U.volScale));
    const v3 cam = ld3(U.camPos), vmin = ld3(U.volMin), vmax = ld3(U.volMax);
    float tEnter = -INFINITY, tExit = INFINITY;
    bool hit = true;
    const float dc[3] = {dn.x, dn.y, dn.z}, cc[3] = {cam.x, cam.y, cam.z};
    for (int a = 0; a < 3; ++a) {
        if (dc[a] == 0.0f) {
            if (cc[a] < U.volMin[a] || cc[a] > U.volMax[a]) hit = false;
            continue;
        }
        const float t0 = (U.volMin[a] - cc[a]) / dc[a];
        const float t1 = (U.volMax[a] - cc[a]) / dc[a];
        tEnter = fmaxf(tEnter, fminf(t0, t1));
        tExit = fminf(tExit, fmaxf(t0, t1));
    }
    const float tStart = fmaxf(tEnter, 0.0f);
    if (!(tExit >= tStart)) hit = false;

    if (hit) {
        v3 rayPos = add(cam, muls(dn, tStart));
        const v3 rayDir = normalize(dn);
        const float jit = jitter[(j & 31) * 32 + (i & 31)];
        rayPos = add(rayPos, muls(muls(rayDir, U.rayStep), jit));
        float inside = inside_count(rayPos, vmin, vmax);
        if (inside >= 3.0f) {
            int curList = 0;  // list * 4 + component
            const int startPush = (i % 2) * kMaxUsage + (j % 2) * kMaxUsage * 2;
            const int stopPush = startPush + kMaxUsage;
            const int maxPerBlock = kMaxUsage * 4;
            const v3 brickRayStep = mul(rayDir, ld3(U.brickStep));
            const v3 rcpDir = rcp_dir<HwApprox>(rayDir);
            const uint2 root = fetch_node(tex, U, 0, 0, 0);
            // octTreeNodePtr is not reset at a restart (GigaVoxels.frag
            // 718-742): a traversal that stops at the root records the
            // previous stopping node's texel.
            uint32_t px = 0, py = 0, pz = 0;
            int nlt = 0, pushed = 0, traversals = 0;
            // A traversal: down from the root to the node the ray stops at,
            // then through that node.  Each is a loop of its own, so that the
            // lanes of a wave meet between them: with both in one loop the
            // lanes that had stopped sampled their bricks while the others'
            // descents waited, and the other way round.
            while (inside >= 3.0f && traversals < U.maxTraversals) {
                uint2 node = root;
                v3 extMin = vmin, extMax = vmax;
                float nodeSize = 1.0f, vh = U.rootVoxelHalf;
                v3 rayBrickPos = rayPos, curBrickRayPos = rayPos;
                uint2 curBrickPtr = root;
                bool loaded, curConst;
                int curDepth = 0, curBrickDepth = 0;
                float hLo, hHi;
                lod_range<HwApprox>(U, rayPos, cam, hLo, hHi);
                for (;;) {
                    curConst = (node.x & kConstBit) != 0u;
                    loaded = (node.x & kResidentBit) != 0u;
                    if (loaded) {
                        curBrickPtr = node;
                        curBrickRayPos = rayBrickPos;
                        curBrickDepth = curDepth;
                    }
                    if (!curConst && !loaded) break;
                    if (!(vh >= hLo && vh <= hHi) && lod_stops(U, rayPos, cam, vh)) break;
                    const uint32_t cx = (node.x >> 20) & 1023u, cy = (node.x >> 10) & 1023u,
                                   cz = node.x & 1023u;
                    // the depth bound never binds for a tree built here (the
                    // last depth has no child pointers); it keeps a damaged
                    // texture from descending forever
                    if ((cx | cy | cz) == 0u || curDepth >= U.depthMinusOne) break;
                    const v3 bo = muls(rayBrickPos, 2.0f);
                    const bool ox = bo.x >= 1.0f, oy = bo.y >= 1.0f, oz = bo.z >= 1.0f;
                    rayBrickPos = mk(ox ? bo.x - 1.0f : bo.x, oy ? bo.y - 1.0f : bo.y,
                                     oz ? bo.z - 1.0f : bo.z);
                    px = cx + (ox ? 1u : 0u);
                    py = cy + (oy ? 1u : 0u);
                    pz = cz + (oz ? 1u : 0u);
                    node = fetch_node(tex, U, px, py, pz);
                    ++curDepth;
                    nodeSize *= 0.5f;
                    extMin = mk(ox ? extMin.x + nodeSize : extMin.x,
                                oy ? extMin.y + nodeSize : extMin.y,
                                oz ? extMin.z + nodeSize : extMin.z);
                    extMax = mk(ox ? extMax.x : extMax.x - nodeSize,
                                oy ? extMax.y : extMax.y - nodeSize,
                                oz ? extMax.z : extMax.z - nodeSize);
                    vh *= 0.5f;
                }
                const uint32_t id = ((px + 1u) << 20) | ((py + 1u) << 10) | (pz + 1u);
                const int n = U.depthMinusOne - (curConst ? curDepth : curBrickDepth);
                const float ratio = ldexpf(1.0f, n);
                const float step = U.rayStep * ratio;
                const int ns = exit_steps(U, rayPos, rayDir, rcpDir, extMin, extMax, n);
                if (curConst) {
                    float cv[4];
                    unpack_rgba(node.y, cv);
                    if (cv[3] < 0.005f) {
                        rayPos = add(rayPos, muls(rayDir, (float)ns * step));   // AdvanceRay
                    } else {
                        const v3 ws = muls(rayDir, step);
                        float src[4];
                        src[3] = 1.0f - pow2n(1.0f - cv[3], n);
                        src[0] = cv[0] * ratio;
                        src[1] = cv[1] * ratio;
                        src[2] = cv[2] * ratio;
                        for (int s = 0; s < ns; ++s) {
                            rayPos = add(rayPos, ws);
                            if (dst[3] > 0.995f) {
                                const int rest = ns - (s + 1);
                                rayPos = add(rayPos, muls(rayDir, (float)rest * step));
                                break;
                            }
                            blend(dst, src);
                        }
                    }
                } else {
                    // the brick's first interior texel (slot origin + 1), in the
                    // pool's normalised coordinates or, in a wide pool, the brick's
                    const v3 bp = U.wide
                        ? ld3(U.firstTexel)
                        : div_pool(U, mk((float)((curBrickPtr.y >> 20) & 1023u),
                                         (float)((curBrickPtr.y >> 10) & 1023u),
                                         (float)(curBrickPtr.y & 1023u)));
                    // (a path with no resident brick keeps the root's word 1,
                    // which need not be a slot: slot 0 is read then, where the
                    // reference reads whatever texel those bits name)
                    const uint32_t slot = curBrickPtr.y < U.wideSlots ? curBrickPtr.y : 0u;
                    gu32 bpool =
                        U.wide ? pool + (uint64_t)slot * (U.pdim[0] * U.pdim[1] * U.pdim[2]) : pool;
                    v3 cbr = add(bp, div_pool(U, mul(curBrickRayPos, ld3(U.brickDim))));
                    const v3 ws = muls(muls(rayDir, U.rayStep), ratio);
                    for (int s = 0; s < ns; ++s) {
                        rayPos = add(rayPos, ws);
                        if (dst[3] > 0.995f) {
                            const int rest = ns - (s + 1);
                            rayPos = add(rayPos, muls(rayDir, (float)rest * step));
                            break;
                        }
                        uint32_t t[8];
                        float w[3];
                        load_sample(bpool, U, cbr, t, w);
                        // eight empty texels add nothing (0 * weight, blended,
                        // unless a weight is no number)
                        if (kOddStep ||
                            (((t[0] | t[1]) | (t[2] | t[3])) | ((t[4] | t[5]) | (t[6] | t[7])))) {
                            float src[4];
                            weigh_sample(t, w, src);
                            src[3] = 1.0f - (1.0f - src[3]);  // pow(1 - a, 1.0)
                            blend(dst, src);
                        }
                        cbr = add(cbr, brickRayStep);
                        if (kOddStep)
                            cbr = mk(cbr.x == cbr.x ? cbr.x : 0.0f, cbr.y == cbr.y ? cbr.y : 0.0f,
                                     cbr.z == cbr.z ? cbr.z : 0.0f);
                    }
                }
                if (nlt >= startPush && nlt < stopPush && pushed < U.maxPush) {
                    ++pushed;
#pragma unroll
                    for (int k = 0; k < kMaxUsage; ++k)
                        if (k == curList) usage[k] = id;
                    curList = curList + 1 == kMaxUsage ? 0 : curList + 1;
                }
                if (dst[3] > 0.995f && (curConst || loaded)) break;
                inside = inside_count(rayPos, vmin, vmax);
                ++traversals;
                ++nlt;
                if (nlt >= maxPerBlock) nlt = 0;
            }
        }
    }
    return hit;
}

// A frame's list of distinct requested node ids.
struct RequestList {
    uint32_t* stamp;              // node texel -> tag of the frame that listed it
    uint32_t* list;
    unsigned long long* times;    // device clock when each was appended
    uint32_t* counts;             // appended (capped), distinct
    uint32_t tag, cap;
};

// Append a wave's node ids of one usage slot to the request list: lanes
// holding the same id elect one leader (ballot loop), leaders claim the node
// texel's frame stamp, the claimants' ids are appended with one count per
// wave.  Every lane of the wave calls it (id 0: none).
__device__ __forceinline__ void append_requests(const RequestList& R, const uint32_t* ndim,
                                                uint32_t id) {
    uint64_t pending = __ballot(id != 0u);
    if (!pending) return;
    const int lane = (int)(threadIdx.x & 63u);
    uint64_t leaders = 0ull;
    while (pending) {
        const int l = __ffsll((unsigned long long)pending) - 1;
        leaders |= 1ull << l;
        pending &= ~__ballot(id == (uint32_t)__builtin_amdgcn_readlane((int)id, l));
    }
    bool claimed = false;
    if ((leaders >> lane) & 1ull) {
        const uint32_t x = ((id >> 20) & 1023u) - 1u;
        const uint32_t y = ((id >> 10) & 1023u) - 1u;
        const uint32_t z = (id & 1023u) - 1u;
        if (x < ndim[0] && y < ndim[1] && z < ndim[2]) {
            const uint32_t t = __umul24(__umul24(z, ndim[1]) + y, ndim[0]) + x;
            // a plain read first: most leaders meet a node another wave has
            // claimed already, and skip the atomic on its (hot) stamp word
            claimed = R.stamp[t] != R.tag && atomicExch(&R.stamp[t], R.tag) != R.tag;
        }
    }
    const uint64_t won = __ballot(claimed);
    if (!won) return;
    const int first = __ffsll((unsigned long long)won) - 1;
    uint32_t base = 0u;
    if (lane == first) base = atomicAdd(&R.counts[1], (uint32_t)__popcll(won));
    base = (uint32_t)__builtin_amdgcn_readlane((int)base, first);
    const uint32_t k = base + (uint32_t)__popcll(won & ((1ull << lane) - 1ull));
    const bool put = claimed && k < R.cap;
    if (put) {
        R.list[k] = id;
        R.times[k] = (unsigned long long)wall_clock64();  // emitted
    }
    const uint64_t kept = __ballot(put);
    if (kept && lane == first) atomicAdd(&R.counts[0], (uint32_t)__popcll(kept));
}

// One octree's frame, one thread per pixel, 16 x 4 pixels a wave and a wave
// per workgroup, so that a wave's place is free again when its own rays end
// (four waves a workgroup: 1.11 ms where this takes 1.05; 8 x 8 pixels:
// 1.06; neighbouring workgroups on one XCD: 1.4 to 1.5, as the rays of one
// part of the image are longer than another's); the wave
// that has cast its pixels lists their distinct node ids itself (the same
// pass over the usage lists in a kernel of its own read 100 MB back at
// 1080p and met few equal ids per wave: 154 us beside a cast of 0.91 ms).
constexpr int kCastW = 16, kCastH = 4;   // pixels of a wave
// Workgroups over w x h pixels; rows of them past a grid's 65536 go on in z.
dim3 cast_grid(uint32_t w, uint32_t h) {
    const uint32_t rows = (h + kCastH - 1) / kCastH, y = std::min(rows, 32768u);
    return dim3((w + kCastW - 1) / kCastW, y, (rows + y - 1) / y);
}
__device__ __forceinline__ int cast_row() {
    return (int)((blockIdx.z * gridDim.y + blockIdx.y) * kCastH + threadIdx.x / kCastW);
}
template <bool kOddStep>
__global__ void __launch_bounds__(kCastW * kCastH)
k_raycast(RayUniforms U, const uint32_t* __restrict__ tex, const uint32_t* __restrict__ pool,
          const float* __restrict__ jitter, uint32_t* __restrict__ rgbaOut,
          float4* __restrict__ rgbaF, uint32_t* __restrict__ usageOut, RequestList R) {
    const int i = U.rx0 + (int)blockIdx.x * kCastW + (int)(threadIdx.x % kCastW);
    const int j = U.ry0 + cast_row();
    uint32_t usage[kMaxUsage];
    if (i < U.rx1 && j < U.ry1) {
        float dst[4];
        cast_pixel<kOddStep>(U, (gu32)tex, (gu32)pool, jitter, i, j, dst, usage);
        const uint64_t pix = (uint64_t)j * U.W + i;
        uint32_t o = 0;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float v = dst[c] * 255.0f;
            v = v > 255.0f ? 255.0f : (v > 0.0f ? v : 0.0f);
            o |= (uint32_t)v << (8 * c);
        }
        rgbaOut[pix] = o;
        rgbaF[pix] = make_float4(dst[0], dst[1], dst[2], dst[3]);  // FragColor
        uint4* u4 = reinterpret_cast<uint4*>(usageOut + pix * kMaxUsage);
        u4[0] = make_uint4(usage[0], usage[1], usage[2], usage[3]);
        u4[1] = make_uint4(usage[4], usage[5], usage[6], usage[7]);
        u4[2] = make_uint4(usage[8], usage[9], usage[10], usage[11]);
    } else {
#pragma unroll
        for (int q = 0; q < kMaxUsage; ++q) usage[q] = 0u;
    }
#pragma unroll
    for (int q = 0; q < kMaxUsage; ++q) append_requests(R, U.ndim, usage[q]);
}

// One octree of a front-to-back frame over several octrees: its uniforms
// and buffers, and the request list its rays append to.
struct TreeCast {
    RayUniforms U;
    const uint32_t* tex;
    const uint32_t* pool;
    RequestList R;
};

// Front to back over n octrees listed in an order every ray meets them in
// (boxes that tile space; the caller's order): each pixel casts its ray
// through every octree whose pixel rectangle holds it, exactly as one
// octree's frame does (cast_pixel), and accumulates the casts' FragColors
// as the renderer's far-to-near blend would (glBlendFunc(GL_SRC_ALPHA,
// GL_ONE_MINUS_SRC_ALPHA) per channel, alpha included): out = sum over
// octrees of T * src * src.a, T the product of (1 - src.a) of the octrees
// before.  A pixel stops once T <= tStop (tStop 0: never, not even at
// T = 0), a wave once all its pixels have; the octrees it skips list no
// requests for it.  With resume the pass continues a frame: acc from frame,
// T from trans (a pass over the octrees in front wrote both); trans, when
// given, receives each pixel's T for the next pass.
template <bool kOddStep>
__global__ void __launch_bounds__(kCastW * kCastH)
k_raycast_multi(const TreeCast* __restrict__ trees, uint32_t n, const float* __restrict__ jitter,
                int32_t W, int32_t x0, int32_t y0, int32_t x1, int32_t y1, float tStop,
                float4* __restrict__ frame, float* __restrict__ trans, int resume) {
    // pixels of the union of the octrees' rectangles, [x0, x1) x [y0, y1)
    const int i = x0 + (int)blockIdx.x * kCastW + (int)(threadIdx.x % kCastW);
    const int j = y0 + cast_row();
    const bool in = i < x1 && j < y1;
    const uint64_t pix = (uint64_t)j * W + i;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    float T = 1.0f;
    if (resume && in) {   // the frame so far, from the octrees in front
        const float4 f = frame[pix];
        acc[0] = f.x;
        acc[1] = f.y;
        acc[2] = f.z;
        acc[3] = f.w;
        T = trans[pix];
    }
    for (uint32_t k = 0; k < n; ++k) {
        const bool want = in && (tStop <= 0.0f || T > tStop);
        if (!__any(want)) break;
        const TreeCast& tc = trees[k];
        const RayUniforms& U = tc.U;
        uint32_t usage[kMaxUsage];
        float dst[4];
        bool act = want && i >= U.rx0 && i < U.rx1 && j >= U.ry0 && j < U.ry1;
        if (act) {
            act = cast_pixel<kOddStep>(U, (gu32)tc.tex, (gu32)tc.pool, jitter, i, j, dst,
                                       usage);
        } else {
#pragma unroll
            for (int q = 0; q < kMaxUsage; ++q) usage[q] = 0u;
        }
        if (act) {
            const float a = dst[3];
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[c] = acc[c] + T * (dst[c] * a);
            T = T * (1.0f - a);
        }
#pragma unroll
        for (int q = 0; q < kMaxUsage; ++q) append_requests(tc.R, U.ndim, usage[q]);
    }
    if (in) {
        frame[pix] = make_float4(acc[0], acc[1], acc[2], acc[3]);
        if (trans) trans[pix] = T;
    }
}

// One caster's pixel rectangle blended into the frame:
// glBlendFunc(GL_SRC_ALPHA, GL_ONE_MINUS_SRC_ALPHA) on an RGBA32F target,
// out = src * src.a + dst * (1 - src.a) for all four channels.
__global__ void k_blend(const float4* __restrict__ src, int32_t W, int32_t x0, int32_t y0,
                        int32_t x1, int32_t y1, float4* __restrict__ dst) {
    const int32_t i = x0 + (int32_t)(blockIdx.x * 16u + (threadIdx.x & 15u));
    const int32_t j = y0 + (int32_t)(blockIdx.y * 16u + (threadIdx.x >> 4));
    if (i >= x1 || j >= y1) return;
    const uint64_t p = (uint64_t)j * W + i;
    const float4 s = src[p], d = dst[p];
    const float a = s.w, k = 1.0f - s.w;
    dst[p] = make_float4(s.x * a + d.x * k, s.y * a + d.y * k, s.z * a + d.z * k,
                         s.w * a + d.w * k);
}

// Jitter table: 32 x 32 values in [0, 1), the k-th from the k+1-th output of
// splitmix64 seeded with `seed` (the state advances by the golden-ratio
// increment, so output k+1 is the finaliser of seed + (k+1) * increment).
__global__ void k_jitter(uint64_t seed, float* __restrict__ out) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= 1024) return;
    uint64_t z = seed + (uint64_t)(k + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    out[k] = (float)(z >> 40) * (1.0f / 16777216.0f);
}

}  // namespace

struct vox_raycaster {
    vox_octree* tree = nullptr;
    bool valid = false;
    int32_t maxW = 0, maxH = 0, W = 0, H = 0;
    uint32_t maxReq = 0, nreq = 0, nreqTotal = 0, tag = 0;
    uint32_t ndim[3] = {0, 0, 0};
    hipStream_t st = nullptr;  // the ray caster's own stream
    DevBuf rgba, rgbaF, usage, req, reqTime, counts, stamp, jitter;
    DevBuf multiTable;          // octree table of front-to-back frames queued here
    // its pinned host staging, two buffers in turn, each reused only after
    // the copy that read it last has run
    void* hostTable[2] = {nullptr, nullptr};
    size_t hostCap[2] = {0, 0};
    hipEvent_t tableCopied[2] = {nullptr, nullptr};
    int tableNext = 0;
    hipEvent_t ev[2] = {nullptr, nullptr};   // round the last frame's cast
    hipEvent_t done = nullptr;  // the last frame's request list is complete
    hipEvent_t read = nullptr;  // a composite has read the last frame
    int32_t rect[4] = {0, 0, 0, 0};  // pixels the last frame wrote
    bool timingPending = false, countsPending = false, haveJitter = false, readPending = false;
    uint64_t jitterSeed = 0;
    double msRay = 0;
    std::stringstream err;
    std::string errCache;
    bool fail(const std::string& m) {
        err << m << std::endl;
        return false;
    }
    bool check(hipError_t e, const char* what) {
        if (e == hipSuccess) return true;
        err << what << " failed: " << hipGetErrorString(e) << std::endl;
        return false;
    }
};

namespace voxmi {

bool raycaster_requests(vox_raycaster* rc, RequestRefs& r) {
    if (!rc || !rc->valid) return false;
    r.ids = rc->req.as<uint32_t>();
    r.times = rc->reqTime.as<uint64_t>();
    r.count = rc->counts.as<uint32_t>();
    r.maxIds = rc->maxReq;
    r.done = rc->done;
    r.tree = rc->tree;
    return true;
}

}  // namespace voxmi

namespace {

}  // namespace

extern "C" {

vox_raycaster* vox_raycaster_create(vox_octree* tree, int32_t max_width, int32_t max_height,
                                    uint32_t max_requests) {
    vox_raycaster* rc = new (std::nothrow) vox_raycaster;
    if (!rc) return nullptr;
    rc->tree = tree;
    OctreeRefs o;
    if (!tree || !octree_refs(tree, o)) {
        rc->fail("raycaster: invalid octree");
        return rc;
    }
    for (int a = 0; a < 3; ++a) rc->ndim[a] = o.ndim[a];
    if (max_width <= 0 || max_height <= 0 || max_requests == 0) {
        rc->fail("raycaster: empty frame or request capacity");
        return rc;
    }
    if (!rc->check(hipStreamCreateWithFlags(&rc->st, hipStreamNonBlocking), "hipStreamCreate"))
        return rc;
    rc->maxW = max_width;
    rc->maxH = max_height;
    rc->maxReq = max_requests;
    const uint64_t npix = (uint64_t)max_width * max_height;
    const uint64_t ntex = (uint64_t)rc->ndim[0] * rc->ndim[1] * rc->ndim[2];
    if (!rc->rgba.ensure(4 * npix, rc->err, "rgba") ||
        !rc->rgbaF.ensure(16 * npix, rc->err, "rgba f32") ||
        !rc->usage.ensure(4 * npix * kMaxUsage, rc->err, "usage") ||
        !rc->req.ensure(4ull * max_requests, rc->err, "requests") ||
        !rc->reqTime.ensure(8ull * max_requests, rc->err, "request times") ||
        !rc->counts.ensure(8, rc->err, "counts") || !rc->stamp.ensure(4 * ntex, rc->err, "stamp") ||
        !rc->jitter.ensure(4 * 1024, rc->err, "jitter"))
        return rc;
    launch_fill_u32(rc->st, rc->stamp.as<uint32_t>(), ntex, 0u);
    launch_fill_u32(rc->st, rc->counts.as<uint32_t>(), 2, 0u);
    for (auto& e : rc->ev)
        if (!rc->check(hipEventCreate(&e), "hipEventCreate")) return rc;
    if (!rc->check(hipEventCreateWithFlags(&rc->read, hipEventDisableTiming), "hipEventCreate") ||
        !rc->check(hipEventCreateWithFlags(&rc->done, hipEventDisableTiming), "hipEventCreate") ||
        !rc->check(hipEventRecord(rc->done, rc->st), "event record") ||
        !rc->check(hipStreamSynchronize(rc->st), "synchronize"))
        return rc;
    rc->valid = true;
    return rc;
}

void vox_raycaster_destroy(vox_raycaster* rc) {
    if (!rc) return;
    if (rc->st) (void)hipStreamSynchronize(rc->st);
    for (auto e : rc->ev)
        if (e) (void)hipEventDestroy(e);
    if (rc->done) (void)hipEventDestroy(rc->done);
    if (rc->read) (void)hipEventDestroy(rc->read);
    rc->rgba.release();
    rc->rgbaF.release();
    rc->usage.release();
    rc->req.release();
    rc->reqTime.release();
    rc->counts.release();
    rc->stamp.release();
    rc->jitter.release();
    rc->multiTable.release();
    for (int b = 0; b < 2; ++b) {
        if (rc->hostTable[b]) (void)hipHostFree(rc->hostTable[b]);
        if (rc->tableCopied[b]) (void)hipEventDestroy(rc->tableCopied[b]);
    }
    if (rc->st) (void)hipStreamDestroy(rc->st);
    delete rc;
}

const char* vox_raycaster_get_error(vox_raycaster* rc) {
    if (!rc) return "null raycaster";
    rc->errCache = rc->err.str();
    return rc->errCache.c_str();
}

namespace {

// Timings of the frame whose events were recorded last (waits for it).
void settle_timing(vox_raycaster* rc) {
    if (!rc->timingPending) return;
    (void)hipEventSynchronize(rc->ev[1]);
    float a = 0;
    (void)hipEventElapsedTime(&a, rc->ev[0], rc->ev[1]);
    rc->msRay = a;
    rc->timingPending = false;
}

}  // namespace

int vox_raycast_frame(vox_raycaster* rc, const vox_camera* cam, const vox_raycast_params* prm) {
    if (!rc || !rc->valid || !cam || !prm) return 0;
    if (cam->width <= 0 || cam->height <= 0 || cam->width > rc->maxW || cam->height > rc->maxH)
        return rc->fail("raycast: viewport exceeds the raycaster's frame size"), 0;
    OctreeRefs o;
    if (!octree_refs(rc->tree, o)) return rc->fail("raycast: octree unavailable"), 0;
    const uint32_t* nd = o.ndim;
    uint32_t* tex = o.tex;
    hipStream_t st = rc->st;
    RayUniforms U;
    if (!ray_uniforms(*cam, *prm, o.levels, o.B, o.poolDims, o.poolWide, o.ndim, U))
        return rc->fail("raycast: empty volume box, ray step below 1e-5 or a pixel rectangle "
                        "outside the viewport"), 0;
    settle_timing(rc);  // the previous frame's events are reused below
    // the node texture and brick pool as the last writer (octree build or
    // brick server frame) left them
    if (!rc->check(hipStreamWaitEvent(st, o.ready, 0), "wait for the node texture")) return 0;
    // a composite still reading the last frame
    if (rc->readPending && !rc->check(hipStreamWaitEvent(st, rc->read, 0), "wait for a composite"))
        return 0;
    rc->readPending = false;
    if (!rc->haveJitter || rc->jitterSeed != prm->jitter_seed) {
        k_jitter<<<4, 256, 0, st>>>(prm->jitter_seed, rc->jitter.as<float>());
        rc->jitterSeed = prm->jitter_seed;
        rc->haveJitter = true;
    }
    rc->W = cam->width;
    rc->H = cam->height;
    const uint32_t rw = (uint32_t)(U.rx1 - U.rx0), rh = (uint32_t)(U.ry1 - U.ry0);
    const uint64_t npix = (uint64_t)rw * rh;
    if (npix * kMaxUsage >= (1ull << 32))
        return rc->fail("raycast: 2^32 usage entries or more"), 0;
    if (++rc->tag == 0) {  // stamp wrap: clear
        launch_fill_u32(st, rc->stamp.as<uint32_t>(), (uint64_t)nd[0] * nd[1] * nd[2], 0u);
        rc->tag = 1;
    }
    launch_fill_u32(st, rc->counts.as<uint32_t>(), 2, 0u);
    (void)hipEventRecord(rc->ev[0], st);
    const dim3 grid = cast_grid(rw, rh);
    const RequestList R{rc->stamp.as<uint32_t>(), rc->req.as<uint32_t>(),
                        rc->reqTime.as<unsigned long long>(), rc->counts.as<uint32_t>(), rc->tag,
                        rc->maxReq};
    const auto cast = U.oddStep ? k_raycast<true> : k_raycast<false>;
    cast<<<grid, kCastW * kCastH, 0, st>>>(U, tex, o.poolCol, rc->jitter.as<float>(),
                                           rc->rgba.as<uint32_t>(), rc->rgbaF.as<float4>(),
                                           rc->usage.as<uint32_t>(), R);
    rc->rect[0] = U.rx0;
    rc->rect[1] = U.ry0;
    rc->rect[2] = U.rx1;
    rc->rect[3] = U.ry1;
    (void)hipEventRecord(rc->ev[1], st);
    if (!rc->check(hipGetLastError(), "raycast kernels") ||
        !rc->check(hipEventRecord(rc->done, st), "event record"))
        return 0;
    rc->timingPending = true;
    rc->countsPending = true;
    return 1;
}

int vox_raycast_frame_multi(vox_raycaster* const* rcs, uint32_t n, const vox_camera* cam,
                            const vox_raycast_params* prms, float* frame, float* transmittance,
                            float t_stop, int32_t resume) {
    if (!rcs || n == 0 || !cam || !prms || !frame || !(t_stop >= 0.0f)) return 0;
    if (resume && !transmittance)
        return rcs[0] ? rcs[0]->fail("raycast multi: resuming needs the transmittance buffer"),
               0 : 0;
    for (uint32_t k = 0; k < n; ++k) {
        if (!rcs[k] || !rcs[k]->valid) return 0;
        for (uint32_t m = 0; m < k; ++m)
            if (rcs[m] == rcs[k]) return rcs[k]->fail("raycast multi: a ray caster appears twice"), 0;
    }
    vox_raycaster* r0 = rcs[0];
    if (cam->width <= 0 || cam->height <= 0) return r0->fail("raycast multi: empty viewport"), 0;
    hipStream_t st = r0->st;
    std::vector<TreeCast> table(n);
    for (uint32_t k = 0; k < n; ++k) {
        vox_raycaster* rc = rcs[k];
        if (cam->width > rc->maxW || cam->height > rc->maxH)
            return rc->fail("raycast multi: viewport exceeds the ray caster's frame size"), 0;
        if (prms[k].jitter_seed != prms[0].jitter_seed)
            return rc->fail("raycast multi: the octrees' jitter seeds differ"), 0;
        OctreeRefs o;
        if (!octree_refs(rc->tree, o)) return rc->fail("raycast multi: octree unavailable"), 0;
        TreeCast& tc = table[k];
        if (!ray_uniforms(*cam, prms[k], o.levels, o.B, o.poolDims, o.poolWide, o.ndim, tc.U))
            return rc->fail("raycast multi: empty volume box, ray step below 1e-5 or a pixel "
                            "rectangle outside the viewport"), 0;
        settle_timing(rc);
        // this octree's node texture and pool as their last writer left them,
        // and its own stream's earlier work
        if (!rc->check(hipStreamWaitEvent(st, o.ready, 0), "wait for the node texture") ||
            (rc != r0 && !rc->check(hipStreamWaitEvent(st, rc->done, 0), "wait for a frame")))
            return 0;
        if (rc->readPending && !rc->check(hipStreamWaitEvent(st, rc->read, 0), "wait for a composite"))
            return 0;
        rc->readPending = false;
        const uint64_t ntex = (uint64_t)rc->ndim[0] * rc->ndim[1] * rc->ndim[2];
        if (++rc->tag == 0) {  // stamp wrap: clear
            launch_fill_u32(st, rc->stamp.as<uint32_t>(), ntex, 0u);
            rc->tag = 1;
        }
        launch_fill_u32(st, rc->counts.as<uint32_t>(), 2, 0u);
        tc.tex = o.tex;
        tc.pool = o.poolCol;
        tc.R = RequestList{rc->stamp.as<uint32_t>(), rc->req.as<uint32_t>(),
                           rc->reqTime.as<unsigned long long>(), rc->counts.as<uint32_t>(),
                           rc->tag, rc->maxReq};
        rc->W = cam->width;
        rc->H = cam->height;
        rc->rect[0] = tc.U.rx0;
        rc->rect[1] = tc.U.ry0;
        rc->rect[2] = tc.U.rx1;
        rc->rect[3] = tc.U.ry1;
    }
    if (!r0->haveJitter || r0->jitterSeed != prms[0].jitter_seed) {
        k_jitter<<<4, 256, 0, st>>>(prms[0].jitter_seed, r0->jitter.as<float>());
        r0->jitterSeed = prms[0].jitter_seed;
        r0->haveJitter = true;
    }
    // a new frame starts cleared (colour 0, transmittance 1); a pass then
    // covers the union of its octrees' rectangles only
    if (!resume) {
        launch_fill_u32(st, reinterpret_cast<uint32_t*>(frame), 4ull * cam->width * cam->height,
                        0u);
        if (transmittance)
            launch_fill_u32(st, reinterpret_cast<uint32_t*>(transmittance),
                            (uint64_t)cam->width * cam->height, 0x3f800000u);  // 1.0f
    }
    int32_t ux0 = cam->width, uy0 = cam->height, ux1 = 0, uy1 = 0;
    for (const TreeCast& tc : table) {
        ux0 = std::min(ux0, tc.U.rx0);
        uy0 = std::min(uy0, tc.U.ry0);
        ux1 = std::max(ux1, tc.U.rx1);
        uy1 = std::max(uy1, tc.U.ry1);
    }
    // the table is copied in stream order, after the previous frame's kernel
    // has read the device copy, from a pinned staging buffer whose last copy
    // has run
    const size_t tbytes = sizeof(TreeCast) * n;
    const int b = r0->tableNext;
    r0->tableNext ^= 1;
    if (!r0->tableCopied[b] &&
        !r0->check(hipEventCreateWithFlags(&r0->tableCopied[b], hipEventDisableTiming),
                   "hipEventCreate"))
        return 0;
    if (!r0->check(hipEventSynchronize(r0->tableCopied[b]), "octree table staging")) return 0;
    if (r0->hostCap[b] < tbytes) {
        if (r0->hostTable[b]) (void)hipHostFree(r0->hostTable[b]);
        r0->hostTable[b] = nullptr;
        r0->hostCap[b] = 0;
        if (!r0->check(hipHostMalloc(&r0->hostTable[b], tbytes, hipHostMallocDefault),
                       "pinned octree table"))
            return 0;
        r0->hostCap[b] = tbytes;
    }
    std::memcpy(r0->hostTable[b], table.data(), tbytes);
    if (!r0->multiTable.ensure(tbytes, r0->err, "octree table") ||
        !r0->check(hipMemcpyAsync(r0->multiTable.p, r0->hostTable[b], tbytes,
                                  hipMemcpyHostToDevice, st),
                   "octree table") ||
        !r0->check(hipEventRecord(r0->tableCopied[b], st), "event record"))
        return 0;
    (void)hipEventRecord(r0->ev[0], st);
    const dim3 grid = cast_grid((uint32_t)(ux1 - ux0), (uint32_t)(uy1 - uy0));
    bool odd = false;
    for (const TreeCast& tc : table) odd = odd || tc.U.oddStep;
    const auto cast = odd ? k_raycast_multi<true> : k_raycast_multi<false>;
    cast<<<grid, kCastW * kCastH, 0, st>>>(r0->multiTable.as<TreeCast>(), n, r0->jitter.as<float>(),
                                           cam->width, ux0, uy0, ux1, uy1, t_stop,
                                           reinterpret_cast<float4*>(frame), transmittance,
                                           resume ? 1 : 0);
    (void)hipEventRecord(r0->ev[1], st);
    if (!r0->check(hipGetLastError(), "raycast multi kernel")) return 0;
    r0->timingPending = true;
    for (uint32_t k = 0; k < n; ++k) {
        if (!rcs[k]->check(hipEventRecord(rcs[k]->done, st), "event record")) return 0;
        rcs[k]->countsPending = true;
    }
    return 1;
}

int vox_composite(vox_raycaster* const* rcs, uint32_t n, float* dst, int32_t width,
                  int32_t height, int32_t clear) {
    if (!dst || width <= 0 || height <= 0 || (n && !rcs)) return 0;
    for (uint32_t k = 0; k < n; ++k) {
        vox_raycaster* rc = rcs[k];
        if (!rc || !rc->valid) return 0;
        if (rc->W != width || rc->H != height)
            return rc->fail("composite: the frame size differs from the ray caster's last frame"), 0;
    }
    // the blends run in the given order on the first caster's stream (the
    // null stream when there is none), after every caster's frame
    hipStream_t st = n ? rcs[0]->st : nullptr;
    for (uint32_t k = 0; k < n; ++k)
        if (hipStreamWaitEvent(st, rcs[k]->done, 0) != hipSuccess) return 0;
    if (clear) launch_fill_u32(st, reinterpret_cast<uint32_t*>(dst), 4ull * width * height, 0u);
    for (uint32_t k = 0; k < n; ++k) {
        const int32_t* r = rcs[k]->rect;
        if (r[2] <= r[0] || r[3] <= r[1]) continue;
        dim3 grid((unsigned)(r[2] - r[0] + 15) / 16, (unsigned)(r[3] - r[1] + 15) / 16);
        k_blend<<<grid, 256, 0, st>>>(rcs[k]->rgbaF.as<float4>(), width, r[0], r[1], r[2], r[3],
                                      reinterpret_cast<float4*>(dst));
    }
    if (hipGetLastError() != hipSuccess) return 0;
    for (uint32_t k = 0; k < n; ++k) {
        if (hipEventRecord(rcs[k]->read, st) != hipSuccess) return 0;
        rcs[k]->readPending = true;
    }
    if (!n && hipStreamSynchronize(st) != hipSuccess) return 0;
    return 1;
}

int vox_raycaster_get_frame(vox_raycaster* rc, vox_frame_view* out) {
    if (!rc || !rc->valid || !out) return 0;
    if (rc->countsPending) {
        uint32_t cnt[2] = {0, 0};
        // the frame may have been cast on another caster's stream (a
        // front-to-back pass); its done event marks the end either way
        if (!rc->check(hipStreamWaitEvent(rc->st, rc->done, 0), "wait for the frame") ||
            !rc->check(hipMemcpyAsync(cnt, rc->counts.p, 8, hipMemcpyDeviceToHost, rc->st),
                       "counts") ||
            !rc->check(hipStreamSynchronize(rc->st), "synchronize"))
            return 0;
        rc->nreq = cnt[0];
        rc->nreqTotal = cnt[1];
        rc->countsPending = false;
    }
    settle_timing(rc);
    out->width = rc->W;
    out->height = rc->H;
    out->rgba = rc->rgba.as<uint32_t>();
    out->rgba_f32 = rc->rgbaF.as<float>();
    out->usage = rc->usage.as<uint32_t>();
    out->requests = rc->req.as<uint32_t>();
    out->nrequests = rc->nreq;
    out->nrequests_total = rc->nreqTotal;
    out->ms_raycast = rc->msRay;
    out->ms_requests = 0.0;   // listed by the cast itself: no time of their own
    return 1;
}

}  // extern "C"
