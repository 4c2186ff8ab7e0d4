// vox_bc.hip -- block compression of the bricks for compressed .gvb output:
// colours as BC3 (DXT5), normals as BC1 (DXT1), each (B+2)^3 brick slice by
// slice in 4x4 blocks.
//
// The reference had the OpenGL driver compress each brick as a 3D S3TC
// texture (VoxelBrickWriter.cu 590-723), so its bytes are driver-specific.
// This encoder is the project's own and deterministic (integer only):
//   endpoints  per-channel max and min of the block's texels, quantized to
//              RGB565 as (v*31+127)/255 and (v*63+127)/255; c0 >= c1;
//   palette    expanded endpoints (q<<3|q>>2, q<<2|q>>4) and the rounded
//              thirds (2a+b+1)/3, (a+2b+1)/3;
//   indices    nearest palette entry in squared RGB distance, lowest index on
//              ties; c0 == c1 gives all indices 0;
//   alpha      a0 = max, a1 = min, entries ((8-k)a0+(k-1)a1+3)/7 for k=2..7,
//              nearest, lowest on ties; a0 == a1 gives all indices 0.
// Blocks of a slice are row-major, slices follow in z (the layout of a
// compressed 3D texture image); texels past the brick edge repeat the edge.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "vox_internal.h"

namespace voxmi {
namespace {

__device__ __forceinline__ uint32_t q5(uint32_t v) { return (v * 31u + 127u) / 255u; }
__device__ __forceinline__ uint32_t q6(uint32_t v) { return (v * 63u + 127u) / 255u; }
__device__ __forceinline__ uint32_t e5(uint32_t q) { return (q << 3) | (q >> 2); }
__device__ __forceinline__ uint32_t e6(uint32_t q) { return (q << 2) | (q >> 4); }

typedef unsigned short us2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ us2 halves(uint32_t v) { return __builtin_bit_cast(us2, v); }

// Channel extremes of a block, two channels to a word: rb holds bytes 0 and 2,
// ga has bytes 1 and 3 in the high bytes of its halves (what lies below them
// cannot change which is larger, so the words are compared as they are).
struct Extremes {
    uint32_t rb0, rb1, ga0, ga1;   // smallest, largest
};
__device__ __forceinline__ Extremes extremes(const uint32_t (&t)[16]) {
    us2 rb0 = halves(0x00ff00ffu), ga0 = halves(0xffffffffu), rb1 = halves(0u), ga1 = rb1;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const us2 rb = halves(t[i] & 0x00ff00ffu), ga = halves(t[i]);
        rb0 = __builtin_elementwise_min(rb0, rb);
        rb1 = __builtin_elementwise_max(rb1, rb);
        ga0 = __builtin_elementwise_min(ga0, ga);
        ga1 = __builtin_elementwise_max(ga1, ga);
    }
    return {__builtin_bit_cast(uint32_t, rb0), __builtin_bit_cast(uint32_t, rb1),
            __builtin_bit_cast(uint32_t, ga0), __builtin_bit_cast(uint32_t, ga1)};
}

// 8-byte colour block of 16 RGB texels (r, g, b in bytes 0..2 of each word).
// The nearest palette entry by squared distance is the one of the largest
// 2 t.P - |P|^2 (|t|^2 is common): one byte dot product an entry, the lowest
// index on ties by its place in the low two bits.
__device__ __forceinline__ uint2 encode_color(const uint32_t (&t)[16], const Extremes& e) {
    uint32_t c0 = (q5(e.rb1 & 255u) << 11) | (q6((e.ga1 >> 8) & 255u) << 5) | q5(e.rb1 >> 16);
    uint32_t c1 = (q5(e.rb0 & 255u) << 11) | (q6((e.ga0 >> 8) & 255u) << 5) | q5(e.rb0 >> 16);
    if (c0 < c1) {
        const uint32_t s = c0;
        c0 = c1;
        c1 = s;
    }
    uint32_t idx = 0u;
    if (c0 != c1) {
        uint32_t P[4][3];
        P[0][0] = e5(c0 >> 11);
        P[0][1] = e6((c0 >> 5) & 63u);
        P[0][2] = e5(c0 & 31u);
        P[1][0] = e5(c1 >> 11);
        P[1][1] = e6((c1 >> 5) & 63u);
        P[1][2] = e5(c1 & 31u);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            P[2][c] = (2u * P[0][c] + P[1][c] + 1u) / 3u;
            P[3][c] = (P[0][c] + 2u * P[1][c] + 1u) / 3u;
        }
        uint32_t pk[4];
        int32_t off[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            pk[k] = P[k][0] | (P[k][1] << 8) | (P[k][2] << 16);   // byte 3 zero: no alpha
            off[k] = 3 - k - 4 * (int32_t)__builtin_amdgcn_udot4(pk[k], pk[k], 0u, false);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            int32_t v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                v[k] = (int32_t)(__builtin_amdgcn_udot4(t[i], pk[k], 0u, false) << 3) + off[k];
            const int32_t best = max(max(v[0], v[1]), max(v[2], v[3]));
            idx |= ((uint32_t)best & 3u) << (2 * i);   // 3 - k
        }
        idx = ~idx;
    }
    return make_uint2(c0 | (c1 << 16), idx);
}

// 8-byte alpha block of 16 alphas (byte 3 of each word).
__device__ __forceinline__ uint2 encode_alpha(const uint32_t (&t)[16], const Extremes& e) {
    const uint32_t a0 = e.ga1 >> 24, a1 = e.ga0 >> 24;
    uint32_t lo = 0u, hi = 0u;   // the indices of 8 texels each
    if (a0 != a1) {
        // eight times the entries: the distances leave room for the index
        uint32_t A[8];
        A[0] = 8u * a0;
        A[1] = 8u * a1;
#pragma unroll
        for (uint32_t k = 2; k < 8u; ++k) A[k] = 8u * (((8u - k) * a0 + (k - 1u) * a1 + 3u) / 7u);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const uint32_t a = (t[i] >> 21) & 0x7f8u;   // 8 alpha
            uint32_t best = 0xffffffffu;
#pragma unroll
            for (uint32_t k = 0; k < 8u; ++k) best = min(best, __builtin_amdgcn_sad_u16(a, A[k], k));
            (i < 8 ? lo : hi) |= (best & 7u) << (3 * (i & 7));
        }
    }
    return make_uint2(a0 | (a1 << 8) | (lo << 16), (lo >> 16) | (hi << 8));
}

constexpr uint32_t kWg = 256;               // blocks a workgroup encodes
constexpr uint32_t kStage = 16u * kWg;      // texels it stages per array, at most

// i / d for a quotient below 2^22, inv = 1 / d: the product is within one.
__device__ __forceinline__ uint32_t div_inv(uint32_t i, uint32_t d, float inv) {
    const uint32_t q = (uint32_t)((float)i * inv);
    const int32_t r = (int32_t)(i - q * d);
    return r < 0 ? q - 1u : (r >= (int32_t)d ? q + 1u : q);
}

// n texels into the LDS, all loads in flight before the first is stored.
template <typename T>
__device__ __forceinline__ void stage(const uint32_t* __restrict__ a,
                                      const uint32_t* __restrict__ b, uint32_t n, uint32_t* la,
                                      uint32_t* lb) {
    constexpr uint32_t per = sizeof(T) / 4u, iters = kStage / (kWg * per);
    const T* ga = reinterpret_cast<const T*>(a);
    const T* gb = reinterpret_cast<const T*>(b);
    T va[iters], vb[iters];
#pragma unroll
    for (uint32_t i = 0; i < iters; ++i) {
        const uint32_t k = i * kWg + threadIdx.x;
        if (k * per < n) {
            va[i] = ga[k];
            vb[i] = gb[k];
        }
    }
#pragma unroll
    for (uint32_t i = 0; i < iters; ++i) {
        const uint32_t k = i * kWg + threadIdx.x;
        if (k * per < n) {
            reinterpret_cast<T*>(la)[k] = va[i];
            reinterpret_cast<T*>(lb)[k] = vb[i];
        }
    }
}

// The 4x4 texels of a block in staged rows of ex texels; rows and columns past
// the slice's edge (`rows` and ex - x0 of them inside) are the edge's again.
// Slices of an even width are pairs of texels at 8-byte addresses.
__device__ __forceinline__ void load_block(const uint32_t* s, uint32_t x0, uint32_t rows,
                                           uint32_t ex, bool pairs, uint32_t (&t)[16]) {
#pragma unroll
    for (uint32_t j = 0; j < 4u; ++j) {
        const uint32_t* row = s + min(j, rows - 1u) * ex;
        if (pairs) {
            const uint2 a = *reinterpret_cast<const uint2*>(row + x0);
            const bool in = x0 + 2u < ex;
            const uint2 b = *reinterpret_cast<const uint2*>(row + (in ? x0 + 2u : x0));
            t[4 * j] = a.x;
            t[4 * j + 1] = a.y;
            t[4 * j + 2] = in ? b.x : a.y;
            t[4 * j + 3] = b.y;   // b is a past the edge
        } else {
#pragma unroll
            for (uint32_t i = 0; i < 4u; ++i) t[4 * j + i] = row[min(x0 + i, ex - 1u)];
        }
    }
}

// Block k of the output from the texels at column x0 of the rows at c and n.
__device__ __forceinline__ void encode_block(const uint32_t* c, const uint32_t* n, uint32_t x0,
                                             uint32_t rows, uint32_t ex, bool pairs, uint64_t k,
                                             uint32_t* __restrict__ outCol,
                                             uint32_t* __restrict__ outNrm) {
    uint32_t t[16];
    load_block(c, x0, rows, ex, pairs, t);
    const Extremes e = extremes(t);
    const uint2 alpha = encode_alpha(t, e);
    const uint2 color = encode_color(t, e);
    reinterpret_cast<uint4*>(outCol)[k] = make_uint4(alpha.x, alpha.y, color.x, color.y);
    load_block(n, x0, rows, ex, pairs, t);
    reinterpret_cast<uint2*>(outNrm)[k] = encode_color(t, extremes(t));
}

// A thread per 4x4 block.  The rows of blocks of all slices of all bricks
// follow each other in memory, so a workgroup takes as many whole ones as 256
// threads hold (perWg, of bxn blocks), and copies their texels, one contiguous
// range, through the LDS: read straight from memory, every load of a wave fell
// into some 50 cache lines.  Bound by VALU issue (4.3 K bricks of 18^3 texels
// of a 512^3 terrain: 142 us with a distance per channel, entry and texel and
// texels read from memory; 130 us with byte dot products, 91 us now).
__global__ __launch_bounds__(kWg) void k_bc_bricks(const uint32_t* __restrict__ col,
                                                   const uint32_t* __restrict__ nrm,
                                                   uint64_t blockRows, uint32_t perWg, uint32_t ex,
                                                   uint32_t ey, double invByn,
                                                   uint32_t* __restrict__ outCol,
                                                   uint32_t* __restrict__ outNrm) {
    __shared__ __align__(8) uint32_t sCol[kStage], sNrm[kStage];
    const uint32_t bxn = (ex + 3u) / 4u, byn = (ey + 3u) / 4u;
    const float invBxn = 1.0f / (float)bxn, invRows = 1.0f / (float)byn;
    const bool pairs = (ex & 1u) == 0u;   // uniform
    const uint32_t lr = div_inv(threadIdx.x, bxn, invBxn), bx = threadIdx.x - lr * bxn;
    for (uint64_t g0 = (uint64_t)blockIdx.x * perWg; g0 < blockRows;
         g0 += (uint64_t)gridDim.x * perWg) {
        const uint32_t n = (uint32_t)min((uint64_t)perWg, blockRows - g0);
        // g0 / byn: (g0 + 1/2) / byn is at least 1 / (2 byn) from a whole
        // number, far above the product's rounding
        const uint64_t slice0 = (uint64_t)(((double)g0 + 0.5) * invByn);
        const uint32_t q0 = (uint32_t)(g0 - slice0 * byn);
        // block row r of the workgroup: its first texel row from the staged first
        auto first = [&](uint32_t r, uint32_t& rows) {
            const uint32_t s = div_inv(q0 + r, byn, invRows), q = q0 + r - s * byn;
            rows = min(4u, ey - 4u * q);
            return s * ey + 4u * q - 4u * q0;
        };
        const uint64_t o = (slice0 * ey + 4u * q0) * ex;
        uint32_t rows;
        const uint32_t lastRow = first(n - 1u, rows), texels = (lastRow + rows) * ex;
        if (pairs) stage<uint2>(col + o, nrm + o, texels, sCol, sNrm);
        else stage<uint32_t>(col + o, nrm + o, texels, sCol, sNrm);
        __syncthreads();
        if (lr < n) {
            const uint32_t at = first(lr, rows) * ex;
            encode_block(sCol + at, sNrm + at, 4u * bx, rows, ex, pairs, g0 * bxn + threadIdx.x,
                         outCol, outNrm);
        }
        __syncthreads();
    }
}

// Bricks of more than 4 kWg texels a row, a row of whose blocks is no
// workgroup's: read from memory as they are.
__global__ __launch_bounds__(kWg) void k_bc_wide(const uint32_t* __restrict__ col,
                                                 const uint32_t* __restrict__ nrm, uint64_t total,
                                                 uint32_t ex, uint32_t ey,
                                                 uint32_t* __restrict__ outCol,
                                                 uint32_t* __restrict__ outNrm) {
    const uint32_t bxn = (ex + 3u) / 4u, byn = (ey + 3u) / 4u;
    for (uint64_t k = blockIdx.x * (uint64_t)kWg + threadIdx.x; k < total;
         k += (uint64_t)gridDim.x * kWg) {
        const uint64_t row = k / bxn, slice = row / byn;
        const uint32_t q = (uint32_t)(row - slice * byn);
        const uint64_t o = (slice * ey + 4u * q) * ex;
        encode_block(col + o, nrm + o, 4u * (uint32_t)(k - row * bxn), min(4u, ey - 4u * q), ex,
                     (ex & 1u) == 0u, k, outCol, outNrm);
    }
}

}  // namespace

uint64_t bc_blocks_per_brick(const uint32_t e[3]) {
    return (uint64_t)((e[0] + 3u) / 4u) * ((e[1] + 3u) / 4u) * e[2];
}

void launch_bc_bricks(hipStream_t st, const uint32_t* col, const uint32_t* nrm, uint64_t nbricks,
                      const uint32_t e[3], uint32_t* outCol, uint32_t* outNrm) {
    const uint32_t bxn = (e[0] + 3u) / 4u, byn = (e[1] + 3u) / 4u;
    const uint64_t blockRows = nbricks * byn * e[2];
    if (blockRows == 0) return;
    auto grid = [](uint64_t items, uint32_t per) {
        return (unsigned)std::min<uint64_t>((items + per - 1u) / per, 1u << 20);
    };
    if (bxn > kWg) {
        k_bc_wide<<<grid(blockRows * bxn, kWg), kWg, 0, st>>>(col, nrm, blockRows * bxn, e[0],
                                                              e[1], outCol, outNrm);
        return;
    }
    const uint32_t perWg = kWg / bxn;
    k_bc_bricks<<<grid(blockRows, perWg), kWg, 0, st>>>(
        col, nrm, blockRows, perWg, e[0], e[1], 1.0 / (double)byn, outCol, outNrm);
}

}  // namespace voxmi
