// The ray cast's arithmetic (voxvizthesis_amd/csrc/vox_raymath.h) for a test on
// the CPU: its shortcuts beside the arithmetic that they stand for.
#include "../../voxvizthesis_amd/csrc/vox_raymath.h"

using namespace voxmi;

namespace {

int g_ulp = 0;   // how far the approximations are off
float moved(float x) {
    for (int k = 0; k < (g_ulp < 0 ? -g_ulp : g_ulp); ++k)
        x = std::nextafter(x, g_ulp < 0 ? 0.0f : INFINITY);
    return x;
}
struct Approx {
    static float rcp(float x) { return moved(1.0f / x); }
    static float rsqrt(float x) { return moved((float)(1.0 / std::sqrt((double)x))); }
    static float sqrt(float x) { return moved(std::sqrt(x)); }
};
v3 at(const float* p, int k) { return {p[3 * k], p[3 * k + 1], p[3 * k + 2]}; }

}  // namespace

extern "C" {

RayUniforms* rm_uniforms(const vox_camera* cam, const vox_raycast_params* prm, int levels,
                         uint32_t brick, uint32_t pool, uint32_t wide) {
    const uint32_t B[3] = {brick, brick, brick}, P[3] = {pool, pool, pool}, n[3] = {64, 64, 64};
    RayUniforms* U = new RayUniforms;
    if (ray_uniforms(*cam, *prm, levels, B, P, wide, n, *U)) return U;
    delete U;
    return nullptr;
}
void rm_free(RayUniforms* U) { delete U; }
int rm_odd_step(const RayUniforms* U) { return (int)U->oddStep; }
void rm_ulp(int ulp) { g_ulp = ulp; }

// n positions in unit-volume coordinates, every level's voxel at each: whether
// the range decides it (to go on), and the test itself (to stop).
void rm_lod(const RayUniforms* U, int n, const float* p, int levels, uint8_t* decided,
            uint8_t* stops) {
    const v3 cam = ld3(U->camPos);
    for (int k = 0; k < n; ++k) {
        float lo, hi, h = U->rootVoxelHalf;
        lod_range<Approx>(*U, at(p, k), cam, lo, hi);
        for (int l = 0; l < levels; ++l, h *= 0.5f) {
            decided[k * levels + l] = h >= lo && h <= hi;
            stops[k * levels + l] = lod_stops(*U, at(p, k), cam, h);
        }
    }
}

// n rays at p along d in boxes [mn, mx], steps of 2^e: the count by products,
// whether that is sure, and the divided count.
void rm_exit(const RayUniforms* U, int n, const float* p, const float* d, const float* mn,
             const float* mx, int e, int* fast, uint8_t* sure, int* divided, int* used) {
    for (int k = 0; k < n; ++k) {
        const v3 dk = at(d, k), rd = rcp_dir<Approx>(dk);
        sure[k] = exit_steps_sure(*U, at(p, k), dk, rd, at(mn, k), at(mx, k), e, fast[k]);
        divided[k] = (int)(exit_time(at(p, k), dk, at(mn, k), at(mx, k)) /
                           (U->rayStep * ldexpf(1.0f, e))) + 1;
        used[k] = exit_steps(*U, at(p, k), dk, rd, at(mn, k), at(mx, k), e);
    }
}

float rm_unorm8_256(uint32_t c) { return unorm8_256(c); }
void rm_div_by(int n, const float* a, float b, float* out) {
    const float r = 1.0f / b;
    for (int k = 0; k < n; ++k) out[k] = div_by(a[k], b, r);
}
// n samples of eight texels and three weights (whole 256ths), and as the sum of
// c / 255 times the weights' products in corner order.
void rm_weigh(int n, const uint32_t* t, const float* w, float* got, float* want) {
    for (int k = 0; k < n; ++k) {
        uint32_t tk[8];
        float wk[3], r[4];
        for (int i = 0; i < 8; ++i) tk[i] = t[8 * k + i];
        for (int i = 0; i < 3; ++i) wk[i] = w[3 * k + i];
        weigh_sample(tk, wk, r);
        for (int c = 0; c < 4; ++c) {
            float s = 0.0f;
            for (int i = 0; i < 8; ++i) {
                float f[3];
                for (int a = 0; a < 3; ++a)
                    f[a] = (i >> a) & 1 ? wk[a] / 256.0f : 1.0f - wk[a] / 256.0f;
                s = s + ((f[0] * f[1]) * f[2]) * ((float)((tk[i] >> (8 * c)) & 255u) / 255.0f);
            }
            got[4 * k + c] = r[c];
            want[4 * k + c] = s;
        }
    }
}

}  // extern "C"
