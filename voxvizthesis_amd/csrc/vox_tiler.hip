// vox_tiler.hip -- assignment of triangles to the 2-D grid of octree tiles
// (C ABI in include/voxmi_tiler.h).
//
// TriangleOctTreeGrid::assignTriangles (main.cu 3986-4030) gives each
// triangle the tiles between the smallest and largest cell its vertices
// reach, where a vertex within the voxel border of a cell edge also reaches
// the neighbouring cell (computeMinMaxGridCell, main.cu 4078-4107) and a
// vertex left of / below the grid origin reaches cell 0.  The lists come out
// in input order, the order the reference appends them in.  Grids of at most
// kLdsTiles tiles are split by counts kept in LDS: every wave owns a run of
// consecutive triangles and counts them per tile, one scan over the (tile,
// wave) counts gives each wave its place in every list, and a second pass
// over the triangles' tile boxes writes them there.  Larger grids write
// (tile, triangle) pairs in triangle order and sort them by tile (stable
// radix sort).
#include <hip/hip_runtime.h>
#include <rocprim/device/device_radix_sort.hpp>

#include <cstdint>
#include <cstring>
#include <new>
#include <sstream>
#include <string>
#include <vector>

#include "../../include/voxmi_tiler.h"
#include "vox_internal.h"

using namespace voxmi;

namespace {

constexpr int kB = 256;

struct Grid {
    float origin[2], size[2], border[2];
    uint32_t dim[2];
};

// computeMinMaxGridCell for one coordinate.
__device__ __forceinline__ void cell_range(float v, float origin, float size, float border,
                                           uint32_t dim, uint32_t& mn, uint32_t& mx) {
    if (v < origin) {
        mn = mx = 0u;
        return;
    }
    const float dist = v - origin;
    const float q = dist / size;
    mn = mx = q < 4294967040.0f ? (uint32_t)q : 0xffffff00u;
    const float maxBorder = (float)(mn + 1u) * size;
    const float d = maxBorder - dist;
    if (d <= border) {
        mx = mn + 1u;
    } else if (mn != 0u) {
        const float minBorder = maxBorder - size;
        if (dist - minBorder <= border) {
            mx = mn;
            mn = mn - 1u;
        }
    }
    if (mn >= dim) mn = dim - 1u;
    if (mx >= dim) mx = dim - 1u;
}

__device__ __forceinline__ void tri_range(const float* __restrict__ v, const Grid& g,
                                          uint32_t& x0, uint32_t& x1, uint32_t& y0, uint32_t& y1) {
    x0 = y0 = 0xffffffffu;
    x1 = y1 = 0u;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        uint32_t a, b, c, d;
        cell_range(v[3 * k], g.origin[0], g.size[0], g.border[0], g.dim[0], a, b);
        cell_range(v[3 * k + 1], g.origin[1], g.size[1], g.border[1], g.dim[1], c, d);
        x0 = a < x0 ? a : x0;
        x1 = b > x1 ? b : x1;
        y0 = c < y0 ? c : y0;
        y1 = d > y1 ? d : y1;
    }
}

// Order-preserving int image of a float (for atomic min / max).
__device__ __forceinline__ int32_t ord(float f) {
    const int32_t i = __float_as_int(f);
    return i >= 0 ? i : (int32_t)(0x80000000u - (uint32_t)i) - 1;
}

// Grids of at most kLdsTiles tiles keep a count per tile and wave and the z
// extents per tile in LDS: 24 bytes per tile and workgroup beside the 9 KB of
// staged vertices, 33 KB at the most, four workgroups (one per SIMD and wave)
// a CU.  There the split takes 137 us for 2 M triangles of a heightfield on 32 x
// 32 tiles and 384 in no order, the sort on 40 x 40 tiles 263 and 693.
constexpr uint32_t kLdsTiles = 1024;
constexpr int kWaves = kB / 64;
// Waves a split is spread over at most: four per SIMD, and the (tile, wave)
// counts it scans are at most 2^22.
constexpr uint64_t kSplitWaves = 4096;

// Tiles of a box, first | last << 16 per axis.
__device__ __forceinline__ uint64_t box_tiles(uint32_t xr, uint32_t yr) {
    return (uint64_t)((xr >> 16) - (xr & 0xffffu) + 1u) * ((yr >> 16) - (yr & 0xffffu) + 1u);
}

__device__ __forceinline__ int32_t wave_min(int32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const int32_t w = __shfl_xor(v, o);
        v = w < v ? w : v;
    }
    return v;
}

// The lanes whose box (xr, yr: first | last << 16) holds tile (x, y).
__device__ __forceinline__ uint64_t lanes_at(bool act, uint32_t xr, uint32_t yr, uint32_t x,
                                             uint32_t y) {
    return __ballot(act && x >= (xr & 0xffffu) && x <= xr >> 16 && y >= (yr & 0xffffu) &&
                    y <= yr >> 16);
}

// Every tile that a wave's triangles reach, once: visit(x, y, m) with m the
// lanes whose box holds it.  Box by box, the lanes with one and the same box
// taken together (neighbouring triangles mostly share theirs; a tile that the
// box of an earlier lane holds has been visited with it), or, where the box round
// them all has no more tiles than the boxes, tile by tile of that one.  From
// kSweep tiles round them all, sweep(x0, x1, y0, y1) over those instead.
template <uint64_t kSweep, class V, class W>
__device__ __forceinline__ void each_tile(bool act, uint32_t xr, uint32_t yr, V visit, W sweep) {
    const uint64_t all = __ballot(act);
    if (!all) return;
    const int f = __ffsll((unsigned long long)all) - 1;
    const uint32_t fx = __builtin_amdgcn_readlane(xr, f), fy = __builtin_amdgcn_readlane(yr, f);
    uint32_t x0 = fx & 0xffffu, x1 = fx >> 16, y0 = fy & 0xffffu, y1 = fy >> 16;
    uint64_t pend = all & ~__ballot(xr == fx && yr == fy);
    if (!pend) {   // one box
        for (uint32_t y = y0; y <= y1; ++y)
            for (uint32_t x = x0; x <= x1; ++x) visit(x, y, all);
        return;
    }
    uint64_t tiles = box_tiles(fx, fy);
    while (pend) {
        const int l = __ffsll((unsigned long long)pend) - 1;
        const uint32_t lx = __builtin_amdgcn_readlane(xr, l);
        const uint32_t ly = __builtin_amdgcn_readlane(yr, l);
        pend &= ~__ballot(xr == lx && yr == ly);
        tiles += box_tiles(lx, ly);
        x0 = min(x0, lx & 0xffffu);
        x1 = max(x1, lx >> 16);
        y0 = min(y0, ly & 0xffffu);
        y1 = max(y1, ly >> 16);
    }
    const uint64_t round = box_tiles(x0 | (x1 << 16), y0 | (y1 << 16));
    if (round >= kSweep) {
        sweep(x0, x1, y0, y1);
        return;
    }
    if (round <= tiles) {
        for (uint32_t y = y0; y <= y1; ++y)
            for (uint32_t x = x0; x <= x1; ++x) {
                const uint64_t m = lanes_at(act, xr, yr, x, y);
                if (m) visit(x, y, m);
            }
        return;
    }
    pend = all;
    while (pend) {
        const int l = __ffsll((unsigned long long)pend) - 1;
        const uint32_t lx = __builtin_amdgcn_readlane(xr, l);
        const uint32_t ly = __builtin_amdgcn_readlane(yr, l);
        pend &= ~__ballot(xr == lx && yr == ly);
        for (uint32_t y = ly & 0xffffu; y <= ly >> 16; ++y)
            for (uint32_t x = lx & 0xffffu; x <= lx >> 16; ++x) {
                const uint64_t m = lanes_at(act, xr, yr, x, y);
                if (!(m & ((1ull << l) - 1ull))) visit(x, y, m);
            }
    }
}

// The counts and z extents of a wave's triangles, by atomics: add(tile, n, lo,
// hi).  Two ways, as atomics in LDS cost less than those in memory.  Either has
// lanes whose boxes few others share walk their own (2 M triangles in no order:
// 0.94 ms a call on 32 x 32 tiles with the lanes of every tile reduced, so
// 0.50; on 40 x 40, in memory, 1.19 and 0.69).
//
// In LDS: the lanes with one and the same box are reduced and its tiles spread
// over the lanes; the rest, or what the first kBoxes boxes leave over, walk.
constexpr int kBoxes = 8, kShared = 8;
template <class F>
__device__ __forceinline__ void count_lds(bool act, uint32_t xr, uint32_t yr, int32_t zlo,
                                          int32_t zhi, uint32_t dimx, F add) {
    const uint32_t lane = threadIdx.x & 63u;
    bool alone = act;
    uint64_t pend = __ballot(act);
    for (int k = 0; k < kBoxes && pend; ++k) {
        const int l = __ffsll((unsigned long long)pend) - 1;
        const uint32_t lx = __builtin_amdgcn_readlane(xr, l);
        const uint32_t ly = __builtin_amdgcn_readlane(yr, l);
        const uint64_t same = __ballot(act && xr == lx && yr == ly);
        pend &= ~same;
        const int n = __popcll(same);
        if (n < kShared) continue;
        const bool in = (same >> lane) & 1ull;
        alone = alone && !in;
        const int32_t lo = wave_min(in ? zlo : 0x7fffffff);
        // the maximum of a as the complement of the minimum of ~a
        const int32_t hi = ~wave_min(in ? ~zhi : 0x7fffffff);
        const uint32_t w = (lx >> 16) - (lx & 0xffffu) + 1u, tiles = (uint32_t)box_tiles(lx, ly);
        for (uint32_t i = lane; i < tiles; i += 64u) {   // at most kLdsTiles
            const uint32_t y = i / w, x = i - y * w;
            add(((ly & 0xffffu) + y) * dimx + (lx & 0xffffu) + x, (uint32_t)n, lo, hi);
        }
    }
    if (alone)
        for (uint32_t y = yr & 0xffffu; y <= yr >> 16; ++y)
            for (uint32_t x = xr & 0xffffu; x <= xr >> 16; ++x) add(y * dimx + x, 1u, zlo, zhi);
}
// In memory: a wave of at most kFew boxes, each of four lanes or more on average,
// has one atomic a tile, any other's lanes walk (2 M triangles of a heightfield
// on 200 x 200 tiles 272 us; with 8 boxes 508, the boxes reduced one by one as in
// LDS 435).
constexpr int kFew = 16;
// Lanes of small boxes look at a tile's extents first: those only widen, so one
// that is wide enough already needs no atomic (2 M triangles in no order on 40 x
// 40 tiles: 0.91 ms without).  Over a large box the looks would be a chain of waits
// that the atomics are not.
constexpr uint32_t kLook = 4;
constexpr uint32_t kFirst = 2048;   // workgroups that start together find nothing set
template <class F>
__device__ __forceinline__ void count_mem(bool act, uint32_t xr, uint32_t yr, int32_t zlo,
                                          int32_t zhi, uint32_t dimx, F add) {
    const uint64_t all = __ballot(act);
    uint64_t pend = all;
    int k = 0;
    for (; k < kFew && pend; ++k) {
        const int l = __ffsll((unsigned long long)pend) - 1;
        pend &= ~__ballot(xr == (uint32_t)__builtin_amdgcn_readlane(xr, l) &&
                          yr == (uint32_t)__builtin_amdgcn_readlane(yr, l));
    }
    if (pend || 4 * k > __popcll(all)) {   // uniform
        const bool look = blockIdx.x >= kFirst && box_tiles(xr, yr) <= kLook;
        if (act)
            for (uint32_t y = yr & 0xffffu; y <= yr >> 16; ++y)
                for (uint32_t x = xr & 0xffffu; x <= xr >> 16; ++x)
                    add(y * dimx + x, 1u, zlo, zhi, look);
        return;
    }
    const uint32_t lane = threadIdx.x & 63u;
    auto visit = [&](uint32_t x, uint32_t y, uint64_t m) {
        const bool in = (m >> lane) & 1ull;
        const int32_t lo = wave_min(in ? zlo : 0x7fffffff);
        const int32_t hi = ~wave_min(in ? ~zhi : 0x7fffffff);
        if (lane == 0u) add(y * dimx + x, (uint32_t)__popcll(m), lo, hi, false);
    };
    each_tile<~0ull>(act, xr, yr, visit, [](uint32_t, uint32_t, uint32_t, uint32_t) {});
}

// First pass of the split: each triangle's tile box (ranges), the triangles
// per (tile, wave), and the tiles' z extents.  Wave w takes the triangles
// [w * per * 64, (w + 1) * per * 64).  Bound by reading the vertices once
// (36 bytes a triangle), which are staged through LDS with 16-byte loads,
// the next 64 triangles' in flight while the current ones are counted.  2.26 M
// triangles on a 4 x 4 grid: 45 us (81 MB of vertices at 1.8 TB/s).
__global__ __launch_bounds__(kB) void k_split_count(const float* __restrict__ verts, uint64_t ntri,
                                                    Grid g, uint32_t n, uint32_t per, uint32_t nw,
                                                    int aligned, uint2* __restrict__ ranges,
                                                    uint32_t* __restrict__ cnt,
                                                    int32_t* __restrict__ zmin,
                                                    int32_t* __restrict__ zmax) {
    extern __shared__ __align__(16) uint32_t lds[];   // kWaves counts per tile, then z extents
    int32_t* s_lo = reinterpret_cast<int32_t*>(lds + kWaves * n);
    int32_t* s_hi = s_lo + n;
    __shared__ __align__(16) float s_v[kWaves][64 * 9];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (uint32_t t = tid; t < n; t += kB) {
#pragma unroll
        for (int k = 0; k < kWaves; ++k) lds[t * kWaves + k] = 0u;
        s_lo[t] = 0x7fffffff;
        s_hi[t] = (int32_t)0x80000000;
    }
    __syncthreads();
    const uint64_t w = (uint64_t)blockIdx.x * kWaves + wv;
    const uint64_t t0 = w * per * 64u, t1 = t0 + (uint64_t)per * 64u < ntri ? t0 + (uint64_t)per * 64u : ntri;
    float* sv = s_v[wv];
    float4 nx[3];
    // 64 triangles are 144 16-byte words (2304 bytes, so the words of a
    // whole group are aligned when the first triangle is)
    auto whole = [&](uint64_t b) { return aligned && b + 64u <= ntri; };
    auto load = [&](uint64_t b) {
        const float4* q = reinterpret_cast<const float4*>(verts + 9 * b);
        nx[0] = q[lane];
        nx[1] = q[64u + lane];
        nx[2] = lane < 16u ? q[128u + lane] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    };
    if (t0 < t1 && whole(t0)) load(t0);
    for (uint64_t b = t0; b < t1; b += 64u) {
        const uint64_t t = b + lane;
        const bool act = t < t1;
        float v[9] = {};
        if (whole(b)) {
            float4* d = reinterpret_cast<float4*>(sv);
            d[lane] = nx[0];
            d[64u + lane] = nx[1];
            if (lane < 16u) d[128u + lane] = nx[2];
            if (b + 64u < t1 && whole(b + 64u)) load(b + 64u);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
#pragma unroll
            for (int k = 0; k < 9; ++k) v[k] = sv[9u * lane + k];
            __builtin_amdgcn_wave_barrier();   // read before the next group's words land
        } else if (act) {
#pragma unroll
            for (int k = 0; k < 9; ++k) v[k] = verts[9 * t + k];
        }
        uint32_t x0 = 0u, x1 = 0u, y0 = 0u, y1 = 0u;
        tri_range(v, g, x0, x1, y0, y1);
        const uint32_t xr = x0 | (x1 << 16), yr = y0 | (y1 << 16);
        if (act) ranges[t] = make_uint2(xr, yr);
        const int32_t zlo = ord(fminf(fminf(v[2], v[5]), v[8]));
        const int32_t zhi = ord(fmaxf(fmaxf(v[2], v[5]), v[8]));
        count_lds(act, xr, yr, zlo, zhi, g.dim[0],
                  [&](uint32_t tile, uint32_t k, int32_t lo, int32_t hi) {
                      atomicAdd(&lds[tile * kWaves + wv], k);
                      atomicMin(&s_lo[tile], lo);
                      atomicMax(&s_hi[tile], hi);
                  });
    }
    __syncthreads();
    for (uint32_t t = tid; t < n; t += kB) {
        const uint4 c = *reinterpret_cast<const uint4*>(lds + t * kWaves);
        *reinterpret_cast<uint4*>(cnt + (uint64_t)t * nw + (uint64_t)blockIdx.x * kWaves) = c;
        if (c.x | c.y | c.z | c.w) {
            atomicMin(&zmin[t], s_lo[t]);
            atomicMax(&zmax[t], s_hi[t]);
        }
    }
}

// Second pass: the wave's places in every tile's list (the scan of its
// counts), handed out in triangle order.  Entries at or past cap are not
// written (the host then grows the lists and runs the pass again).  A wave
// goes tile by tile, each a read and a write of a place that the next waits for,
// or, over kSweepTiles tiles and more, a lane takes a tile and its triangles one
// after the other (100 triangles in no order on 934 tiles 60 us and 19; 2 M on 32 x
// 32 tiles 0.50 ms a call and 0.39; swept from 16 tiles on, 4 x 4 tiles take 205 us
// for 153).
constexpr uint64_t kSweepTiles = 32;
__global__ __launch_bounds__(kB) void k_split_write(const uint2* __restrict__ ranges, uint64_t ntri,
                                                    uint32_t dimx, uint32_t n, uint32_t per,
                                                    uint32_t nw, const uint32_t* __restrict__ excl,
                                                    uint64_t cap, uint32_t* __restrict__ tris) {
    extern __shared__ __align__(16) uint32_t lds[];   // next place per (tile, wave)
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (uint32_t t = tid; t < n; t += kB)
        *reinterpret_cast<uint4*>(lds + t * kWaves) = *reinterpret_cast<const uint4*>(
            excl + (uint64_t)t * nw + (uint64_t)blockIdx.x * kWaves);
    __syncthreads();
    const uint64_t w = (uint64_t)blockIdx.x * kWaves + wv;
    const uint64_t t0 = w * per * 64u, t1 = t0 + (uint64_t)per * 64u < ntri ? t0 + (uint64_t)per * 64u : ntri;
    volatile uint32_t* place = lds;            // lane 0 moves it on, every lane reads it
    uint2 r = t0 + lane < t1 ? ranges[t0 + lane] : make_uint2(0u, 0u);
    for (uint64_t b = t0; b < t1; b += 64u) {
        const uint64_t t = b + lane;
        const bool act = t < t1;
        const uint2 cur = r;
        if (t + 64u < t1) r = ranges[t + 64u];
        auto visit = [&](uint32_t x, uint32_t y, uint64_t m) {
            const uint32_t tile = y * dimx + x;
            const uint32_t at = place[tile * kWaves + wv];
            const uint64_t o = (uint64_t)at + (uint64_t)__popcll(m & ((1ull << lane) - 1ull));
            if (((m >> lane) & 1ull) && o < cap) tris[o] = (uint32_t)t;
            __builtin_amdgcn_wave_barrier();
            if (lane == 0u) place[tile * kWaves + wv] = at + (uint32_t)__popcll(m);
            __builtin_amdgcn_wave_barrier();
        };
        auto sweep = [&](uint32_t x0, uint32_t x1, uint32_t y0, uint32_t y1) {
            const uint32_t w = x1 - x0 + 1u, tiles = w * (y1 - y0 + 1u);   // at most kLdsTiles
            for (uint32_t i0 = 0; i0 < tiles; i0 += 64u) {
                // the triangles whose boxes reach these 64 tiles' rows and, in
                // one row, columns
                const uint32_t i1 = min(i0 + 63u, tiles - 1u), ya = i0 / w, yb = i1 / w;
                const uint32_t xa = ya == yb ? x0 + i0 - ya * w : x0;
                const uint32_t xb = ya == yb ? x0 + i1 - yb * w : x1;
                uint64_t left = __ballot(act && (cur.x & 0xffffu) <= xb && cur.x >> 16 >= xa &&
                                         (cur.y & 0xffffu) <= y0 + yb && cur.y >> 16 >= y0 + ya);
                if (!left) continue;
                const uint32_t i = i0 + lane, dy = i / w, x = x0 + i - dy * w, y = y0 + dy;
                const uint32_t tile = i < tiles ? y * dimx + x : 0u;
                uint32_t at = place[tile * kWaves + wv];
                for (; left; left &= left - 1ull) {
                    const int l = __ffsll((unsigned long long)left) - 1;
                    const uint32_t lx = __builtin_amdgcn_readlane(cur.x, l);
                    const uint32_t ly = __builtin_amdgcn_readlane(cur.y, l);
                    if (i < tiles && x >= (lx & 0xffffu) && x <= lx >> 16 && y >= (ly & 0xffffu) &&
                        y <= ly >> 16) {
                        if (at < cap) tris[at] = (uint32_t)(b + (uint32_t)l);
                        ++at;
                    }
                }
                if (i < tiles) place[tile * kWaves + wv] = at;
                __builtin_amdgcn_wave_barrier();   // other lanes read it next
            }
        };
        each_tile<kSweepTiles>(act, cur.x, cur.y, visit, sweep);
    }
}

// Counts per tile and per triangle, and the tiles' z extents (grids of more
// than kLdsTiles tiles).  Bound by the atomics: with one per lane and extent,
// 2.26 M triangles on a 4 x 4 grid took 28.4 ms.
__global__ void k_tile_count(const float* __restrict__ verts, uint64_t ntri, Grid g,
                             uint32_t* __restrict__ cnt, uint32_t* __restrict__ triCnt,
                             int32_t* __restrict__ zmin, int32_t* __restrict__ zmax) {
    const uint64_t t = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    const bool act0 = t < ntri;
    if (!__ballot(act0)) return;   // whole waves: every lane takes part below
    float v[9] = {};
    if (act0) {
#pragma unroll
        for (int k = 0; k < 9; ++k) v[k] = verts[9 * t + k];
    }
    uint32_t x0, x1, y0, y1;
    tri_range(v, g, x0, x1, y0, y1);
    if (act0) triCnt[t] = (x1 - x0 + 1u) * (y1 - y0 + 1u);
    const int32_t zlo = ord(fminf(fminf(v[2], v[5]), v[8]));
    const int32_t zhi = ord(fmaxf(fmaxf(v[2], v[5]), v[8]));
    count_mem(act0, x0 | (x1 << 16), y0 | (y1 << 16), zlo, zhi, g.dim[0],
              [&](uint32_t tile, uint32_t k, int32_t lo, int32_t hi, bool look) {
                  atomicAdd(&cnt[tile], k);
                  bool low = true, high = true;
                  if (look) {
                      low = lo < __hip_atomic_load(&zmin[tile], __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_WORKGROUP);
                      high = hi > __hip_atomic_load(&zmax[tile], __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_WORKGROUP);
                  }
                  if (low) atomicMin(&zmin[tile], lo);
                  if (high) atomicMax(&zmax[tile], hi);
              });
}

// The (tile, triangle) pairs of triangle t at its offset: pairs in
// triangle order, tiles row by row within a triangle.
__global__ void k_tile_pairs(const float* __restrict__ verts, uint64_t ntri, Grid g,
                             const uint32_t* __restrict__ triOff, uint32_t* __restrict__ keys,
                             uint32_t* __restrict__ vals) {
    const uint64_t t = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (t >= ntri) return;
    uint32_t x0, x1, y0, y1;
    tri_range(verts + 9 * t, g, x0, x1, y0, y1);
    uint32_t o = triOff[t];
    for (uint32_t y = y0; y <= y1; ++y)
        for (uint32_t x = x0; x <= x1; ++x) {
            keys[o] = y * g.dim[0] + x;
            vals[o] = (uint32_t)t;
            ++o;
        }
}

__global__ void k_z_init(uint64_t n, int32_t* __restrict__ zmin, int32_t* __restrict__ zmax) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x) {
        zmin[i] = 0x7fffffff;
        zmax[i] = (int32_t)0x80000000;
    }
}

__device__ __forceinline__ float unord(int32_t o) {
    return __int_as_float(o >= 0 ? o : (int32_t)(0x80000000u - (uint32_t)(o + 1)));
}

__global__ void k_unord(uint64_t n, const int32_t* __restrict__ zmin,
                        const int32_t* __restrict__ zmax, float* __restrict__ zminf,
                        float* __restrict__ zmaxf) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x) {
        zminf[i] = unord(zmin[i]);
        zmaxf[i] = unord(zmax[i]);
    }
}

// The lists' starts from the scanned (tile, wave) counts, and the z extents
// as floats.
__global__ void k_split_finish(uint32_t n, uint32_t nw, const uint32_t* __restrict__ excl,
                               const int32_t* __restrict__ zmin, const int32_t* __restrict__ zmax,
                               uint32_t* __restrict__ start, float* __restrict__ zminf,
                               float* __restrict__ zmaxf) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t > n) return;
    start[t] = excl[(uint64_t)t * nw];   // excl[n * nw] is the scan's total
    if (t == n) return;
    zminf[t] = unord(zmin[t]);
    zmaxf[t] = unord(zmax[t]);
}

// For every tile and group boundary k: the position in the tile's ordered
// list of its first triangle with index >= first[k].
__global__ void k_group_bounds(const uint32_t* __restrict__ start, const uint32_t* __restrict__ tris,
                               uint64_t ntiles, const uint32_t* __restrict__ first, uint32_t nb,
                               uint32_t* __restrict__ out) {
    const uint64_t total = ntiles * nb;
    for (uint64_t e = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; e < total;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t tile = e / nb;
        const uint32_t v = first[e - tile * nb];
        uint32_t lo = start[tile], hi = start[tile + 1];
        while (lo < hi) {
            const uint32_t mid = lo + ((hi - lo) >> 1);
            if (tris[mid] < v) lo = mid + 1;
            else hi = mid;
        }
        out[e] = lo;
    }
}

unsigned grid_for(uint64_t n) {
    const uint64_t g = (n + kB - 1) / kB;
    return (unsigned)(g < 65536 ? (g ? g : 1) : 65536);
}

}  // namespace

struct vox_tiler {
    bool valid = false;
    hipStream_t st = nullptr;
    uint64_t ntiles = 0, pairs = 0;
    DevBuf cnt, start, tris, zmin, zmax, zminf, zmaxf, scanTmp, hostVerts;
    DevBuf triCnt, triOff, triScan, keys, keys2, vals, sortTmp;
    DevBuf ranges, waveCnt, waveExcl;   // the LDS split's tile boxes and counts
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

namespace {

// Tile lists by the LDS split (ntri > 0, n <= kLdsTiles).
bool assign_split(vox_tiler* t, const float* verts, uint64_t ntri, const Grid& g, uint32_t n) {
    hipStream_t st = t->st;
    // 64-triangle groups per wave
    const uint32_t per = (uint32_t)((ntri + 64 * kSplitWaves - 1) / (64 * kSplitWaves));
    const uint32_t blocks = (uint32_t)((ntri + 64ull * per * kWaves - 1) / (64ull * per * kWaves));
    const uint32_t nw = blocks * kWaves;
    const uint64_t m = (uint64_t)n * nw;
    // most triangles lie in one tile: room for a quarter more entries than
    // triangles, so that the lists' size is only looked at once they are written
    if (!t->ranges.ensure(8 * ntri, t->err, "tile boxes") ||
        !t->waveCnt.ensure(4 * m, t->err, "tile counts") ||
        !t->waveExcl.ensure(4 * (m + 1), t->err, "tile offsets") ||
        !ensure_scan_tmp(t->scanTmp, m, st, t->err, "scan") ||
        !t->tris.ensure(4 * (ntri + ntri / 4) + 1024, t->err, "tile triangles"))
        return false;
    const int aligned = (reinterpret_cast<uintptr_t>(verts) & 15u) == 0 ? 1 : 0;
    k_split_count<<<blocks, kB, 4 * (kWaves + 2) * n, st>>>(
        verts, ntri, g, n, per, nw, aligned, t->ranges.as<uint2>(), t->waveCnt.as<uint32_t>(),
        t->zmin.as<int32_t>(), t->zmax.as<int32_t>());
    launch_scan(st, t->waveCnt.as<uint32_t>(), t->waveExcl.as<uint32_t>(), m,
                t->scanTmp.as<uint32_t>());
    k_split_finish<<<(n + kB) / kB, kB, 0, st>>>(n, nw, t->waveExcl.as<uint32_t>(),
                                                 t->zmin.as<int32_t>(), t->zmax.as<int32_t>(),
                                                 t->start.as<uint32_t>(), t->zminf.as<float>(),
                                                 t->zmaxf.as<float>());
    uint32_t total = 0;
    for (int pass = 0; pass < 2; ++pass) {
        const uint64_t cap = t->tris.cap / 4;
        k_split_write<<<blocks, kB, 4 * kWaves * n, st>>>(t->ranges.as<uint2>(), ntri, g.dim[0], n,
                                                          per, nw, t->waveExcl.as<uint32_t>(), cap,
                                                          t->tris.as<uint32_t>());
        if (!t->check(hipGetLastError(), "tiler kernels") ||
            !t->check(hipMemcpyAsync(&total, t->start.as<uint32_t>() + n, 4, hipMemcpyDeviceToHost,
                                     st),
                      "pairs") ||
            !t->check(hipStreamSynchronize(st), "synchronize"))
            return false;
        if (total <= cap) break;
        if (!t->tris.ensure(4ull * total, t->err, "tile triangles")) return false;
    }
    t->pairs = total;
    return true;
}

// Tile lists by sorting (tile, triangle) pairs.
bool assign_sort(vox_tiler* t, const float* verts, uint64_t ntri, const Grid& g, uint64_t n) {
    hipStream_t st = t->st;
    const uint64_t nt = ntri ? ntri : 1;
    if (!t->cnt.ensure(4 * (n + 1), t->err, "tile counts") ||
        !ensure_scan_tmp(t->scanTmp, n, st, t->err, "scan") ||
        !t->triCnt.ensure(4 * (nt + 1), t->err, "triangle counts") ||
        !t->triOff.ensure(4 * (nt + 1), t->err, "triangle offsets") ||
        !ensure_scan_tmp(t->triScan, nt, st, t->err, "scan"))
        return false;
    launch_fill_u32(st, t->cnt.as<uint32_t>(), n, 0u);
    if (ntri) {
        k_tile_count<<<(unsigned)((ntri + kB - 1) / kB), kB, 0, st>>>(
            verts, ntri, g, t->cnt.as<uint32_t>(), t->triCnt.as<uint32_t>(),
            t->zmin.as<int32_t>(), t->zmax.as<int32_t>());
        launch_scan(st, t->triCnt.as<uint32_t>(), t->triOff.as<uint32_t>(), ntri,
                    t->triScan.as<uint32_t>());
    }
    launch_scan(st, t->cnt.as<uint32_t>(), t->start.as<uint32_t>(), n, t->scanTmp.as<uint32_t>());
    uint32_t total = 0;
    if (!t->check(hipMemcpyAsync(&total, t->start.as<uint32_t>() + n, 4, hipMemcpyDeviceToHost, st),
                  "pairs") ||
        !t->check(hipStreamSynchronize(st), "synchronize"))
        return false;
    t->pairs = total;
    if (!t->tris.ensure(4ull * total + 4, t->err, "tile triangles")) return false;
    if (total) {
        if (!t->keys.ensure(4ull * total, t->err, "pair keys") ||
            !t->keys2.ensure(4ull * total, t->err, "pair keys") ||
            !t->vals.ensure(4ull * total, t->err, "pair triangles"))
            return false;
        k_tile_pairs<<<(unsigned)((ntri + kB - 1) / kB), kB, 0, st>>>(
            verts, ntri, g, t->triOff.as<uint32_t>(), t->keys.as<uint32_t>(),
            t->vals.as<uint32_t>());
        unsigned bits = 1;
        while (bits < 32 && (1ull << bits) < n) ++bits;
        size_t tmpBytes = 0;
        if (!t->check(rocprim::radix_sort_pairs(nullptr, tmpBytes, t->keys.as<uint32_t>(),
                                                t->keys2.as<uint32_t>(), t->vals.as<uint32_t>(),
                                                t->tris.as<uint32_t>(), (size_t)total, 0u, bits,
                                                st),
                      "sort size") ||
            !t->sortTmp.ensure(tmpBytes, t->err, "sort storage") ||
            !t->check(rocprim::radix_sort_pairs(t->sortTmp.p, tmpBytes, t->keys.as<uint32_t>(),
                                                t->keys2.as<uint32_t>(), t->vals.as<uint32_t>(),
                                                t->tris.as<uint32_t>(), (size_t)total, 0u, bits,
                                                st),
                      "sort"))
            return false;
    }
    k_unord<<<grid_for(n), kB, 0, st>>>(n, t->zmin.as<int32_t>(), t->zmax.as<int32_t>(),
                                        t->zminf.as<float>(), t->zmaxf.as<float>());
    return t->check(hipGetLastError(), "tiler kernels") &&
           t->check(hipStreamSynchronize(st), "synchronize");
}

}  // namespace

extern "C" {

vox_tiler* vox_tiler_create(void) {
    vox_tiler* t = new (std::nothrow) vox_tiler;
    if (!t) return nullptr;
    if (!t->check(hipStreamCreateWithFlags(&t->st, hipStreamNonBlocking), "hipStreamCreate"))
        return t;
    t->valid = true;
    return t;
}

void vox_tiler_destroy(vox_tiler* t) {
    if (!t) return;
    if (t->st) (void)hipStreamSynchronize(t->st);
    DevBuf* b[] = {&t->cnt, &t->start, &t->tris, &t->zmin, &t->zmax, &t->zminf, &t->zmaxf,
                   &t->scanTmp, &t->hostVerts, &t->triCnt, &t->triOff, &t->triScan, &t->keys,
                   &t->keys2, &t->vals, &t->sortTmp, &t->ranges, &t->waveCnt, &t->waveExcl};
    for (DevBuf* x : b) x->release();
    if (t->st) (void)hipStreamDestroy(t->st);
    delete t;
}

const char* vox_tiler_get_error(vox_tiler* t) {
    if (!t) return "null tiler";
    t->errCache = t->err.str();
    return t->errCache.c_str();
}

int vox_tiler_assign(vox_tiler* t, const float* verts, uint64_t ntri, int32_t device,
                     const vox_tile_grid* grid) {
    if (!t || !t->valid || !grid) return 0;
    if (ntri && !verts) return t->fail("tiler: no vertices"), 0;
    if (ntri && !device) {
        if (!t->hostVerts.ensure(36 * ntri, t->err, "vertices") ||
            !t->check(hipMemcpyAsync(t->hostVerts.p, verts, 36 * ntri, hipMemcpyHostToDevice, t->st),
                      "vertex upload"))
            return 0;
        verts = t->hostVerts.as<float>();
    }
    Grid g;
    for (int a = 0; a < 2; ++a) {
        g.origin[a] = grid->origin[a];
        g.size[a] = grid->size[a];
        g.border[a] = grid->border[a];
        g.dim[a] = grid->dim[a];
        if (!(g.size[a] > 0.0f) || g.dim[a] == 0 || g.dim[a] > 65536)
            return t->fail("tiler: bad grid"), 0;
    }
    const uint64_t n = (uint64_t)g.dim[0] * g.dim[1];
    if (n >= 0xffffffffull) return t->fail("tiler: too many tiles"), 0;
    t->ntiles = n;
    hipStream_t st = t->st;
    if (!t->start.ensure(4 * (n + 1), t->err, "tile offsets") ||
        !t->zmin.ensure(4 * n, t->err, "z min") || !t->zmax.ensure(4 * n, t->err, "z max") ||
        !t->zminf.ensure(4 * n, t->err, "z min") || !t->zmaxf.ensure(4 * n, t->err, "z max"))
        return 0;
    k_z_init<<<grid_for(n), kB, 0, st>>>(n, t->zmin.as<int32_t>(), t->zmax.as<int32_t>());
    // The split through LDS wherever the tiles' counters fit there (2.26 M
    // triangles on a 4 x 4 grid: 103 us a call; the sort's pairs, its three
    // passes and their scans alone took 100 us of device time beside the
    // count); the sort beyond.
    return (ntri && n <= kLdsTiles ? assign_split(t, verts, ntri, g, (uint32_t)n)
                                   : assign_sort(t, verts, ntri, g, n))
               ? 1
               : 0;
}

int vox_tiler_group_bounds(vox_tiler* t, const uint32_t* first, uint32_t nbounds, uint32_t* out) {
    if (!t || !t->valid || !first || !out || nbounds == 0) return 0;
    if (t->ntiles == 0) return t->fail("tiler: assign first"), 0;
    const uint64_t total = t->ntiles * nbounds;
    DevBuf f, o;
    bool ok = f.ensure(4ull * nbounds, t->err, "bounds") && o.ensure(4 * total, t->err, "bounds") &&
              t->check(hipMemcpyAsync(f.p, first, 4ull * nbounds, hipMemcpyHostToDevice, t->st),
                       "bounds upload");
    if (ok) {
        k_group_bounds<<<grid_for(total), kB, 0, t->st>>>(t->start.as<uint32_t>(),
                                                          t->tris.as<uint32_t>(), t->ntiles,
                                                          f.as<uint32_t>(), nbounds,
                                                          o.as<uint32_t>());
        ok = t->check(hipGetLastError(), "bounds kernel") &&
             t->check(hipMemcpyAsync(out, o.p, 4 * total, hipMemcpyDeviceToHost, t->st),
                      "bounds") &&
             t->check(hipStreamSynchronize(t->st), "synchronize");
    }
    f.release();
    o.release();
    return ok ? 1 : 0;
}

int vox_tiler_get(vox_tiler* t, vox_tile_lists* out) {
    if (!t || !t->valid || !out) return 0;
    out->ntiles = t->ntiles;
    out->pairs = t->pairs;
    out->tile_start = t->start.as<uint32_t>();
    out->tile_tris = t->tris.as<uint32_t>();
    out->tile_zmin = t->zminf.as<float>();
    out->tile_zmax = t->zmaxf.as<float>();
    return 1;
}

}  // extern "C"
