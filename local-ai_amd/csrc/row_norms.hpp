// What the RMS norms of f16 rows share: layer_glue.hip has them on their own, row_norms.hip behind a product.
#pragma once
#include "common.hpp"

namespace {

// Sum over a workgroup of up to 256 threads (4 waves).
__device__ __forceinline__ float block_sum(float v, float* scratch, uint32_t threads) {
    v = lh_group_sum(v, 64);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwaves = (threads + 63) >> 6;
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    float t = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; w++) t = w < nwaves ? t + scratch[w] : t;
    __syncthreads();
    return t;
}

__device__ __forceinline__ float norm_tail(float normed, float res, uint32_t tail, float scale) { return lh_norm_tail(normed, res, tail, scale); }

// The arithmetic of one 8-element chunk, shared by every kernel that must reproduce the stand-alone norm bit for bit.
__device__ __forceinline__ void rms_sumsq8(const uint4& v, float& s) {
    const uint32_t wv[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int j = 0; j < 4; j++) { const float a = lh_h2f((uint16_t)(wv[j] & 0xFFFF)), b = lh_h2f((uint16_t)(wv[j] >> 16)); s += a * a; s += b * b; }
}
template <bool ADD>
__device__ __forceinline__ uint4 rms_apply8(const uint4& v, const uint4& g, const uint4& r, float rms, uint32_t tail, float scale) {
    const uint32_t wv[4] = {v.x, v.y, v.z, v.w}, wg[4] = {g.x, g.y, g.z, g.w}, wr[4] = {r.x, r.y, r.z, r.w};
    uint32_t wo[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        float lo = lh_norm_product(lh_h2f((uint16_t)(wv[j] & 0xFFFF)), rms, lh_h2f((uint16_t)(wg[j] & 0xFFFF)));
        float hi = lh_norm_product(lh_h2f((uint16_t)(wv[j] >> 16)), rms, lh_h2f((uint16_t)(wg[j] >> 16)));
        if (ADD) {
            const float rlo = lh_h2f((uint16_t)(wr[j] & 0xFFFF)), rhi = lh_h2f((uint16_t)(wr[j] >> 16));
            if (tail) { lo = norm_tail(lo, rlo, tail, scale); hi = norm_tail(hi, rhi, tail, scale); }
            else { lo += rlo; hi += rhi; }
        }
        wo[j] = (uint32_t)lh_f2h_exact(lo) | ((uint32_t)lh_f2h_exact(hi) << 16);
    }
    return make_uint4(wo[0], wo[1], wo[2], wo[3]);
}

// Eight values as scale_in_place_gpu_into leaves them.
__device__ __forceinline__ uint4 scale8(uint4 v, float by) {
    uint32_t* w = &v.x;
#pragma unroll
    for (int j = 0; j < 4; j++) w[j] = (uint32_t)lh_f2h(lh_h2f((uint16_t)(w[j] & 0xFFFF)) * by) | ((uint32_t)lh_f2h(lh_h2f((uint16_t)(w[j] >> 16)) * by) << 16);
    return v;
}

}  // namespace
