// The norms of rows that a product leaves as partial tiles, with what surrounds them in a layer (layer_glue.hip has each step on its own).  A file of its own
// because its kernel's first arguments arrive in registers with the wave (see the Makefile): 0.1 us less for it, 0.13 more for a residual addition.
#include "row_norms.hpp"
#include <type_traits>

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// rms_norm_kernel<ADD, 8> with its input taken either from f16 rows or from the f32 partial tiles of a k-split product
// (summed in split order and rounded to f16, which is what the product's own reduction would have stored), optionally
// followed by the output scale (scale_in_place.metal:5-14) and by a second plain norm of the row just produced
// (layer.rs:640-652: post-attention norm + residual, then the feed-forward norm): up to four dispatches of a decode
// batch's layer in one.  Same thread count, accumulation order and rounding points as the separate kernels, so the
// results are theirs bit for bit.  A thread keeps its (two, or up to four) 8-element chunks in registers between the passes.
// A chain on one CU, bound by its trips to memory: with the loads under conditions the compiler had put five of them one behind the other,
// and code for four chunks and every tail took more instruction fetches.  64 rows of 1536 (of 1024: 16), two norms, 1, 2, 3, 6, 8 and 16 splits: 4.0, 4.2, 4.5, 5.5, 6.2 and
// 7.8 us, now 3.6, 3.6, 3.6, 4.1, 4.7 and 6.0 (a trip for three splits; a product of 64 rows has 6 or 8 in most layers, one of 256 rows 2 or 3).
template <bool PART, bool ADD, int CHUNKS>
__global__ __launch_bounds__(256) void rms_norm_fused_kernel(const uint16_t* nw, const uint16_t* res, const uint16_t* nw2, const float* partial, uint32_t dim, uint32_t splits,
                                                            uint32_t part_rows, uint32_t part_cols, uint32_t threads, const LhNormFused a) {
    __shared__ float scratch[4];
    const uint32_t rowi = blockIdx.x;
    const size_t row = (size_t)rowi * dim;
    uint4 x[CHUNKS], o[CHUNKS];
    // The norm weights, the residual and the second norm's weights are requested here, with the row itself: read where they
    // are used, each waits for memory again behind the barrier of the pass before.  A thread without a chunk reads its row's
    // first: with a branch around them, the values it would leave alone are put in place behind the loads, and those waited for.
    const uint16_t* const second = nw2 != nullptr ? nw2 : nw;
    bool has[CHUNKS];
    uint32_t at[CHUNKS];
    uint4 gw[CHUNKS], rr[CHUNKS], gw2[CHUNKS];
#pragma unroll
    for (int it = 0; it < CHUNKS; it++) {
        const uint32_t i = (threadIdx.x + it * threads) * 8;
        has[it] = i < dim;
        at[it] = has[it] ? i : 0u;
        gw[it] = *reinterpret_cast<const uint4*>(nw + at[it]);
        if (ADD) rr[it] = *reinterpret_cast<const uint4*>(res + row + at[it]);
        gw2[it] = *reinterpret_cast<const uint4*>(second + at[it]);
    }
    if constexpr (PART) {
        // the splits of two chunks, three at a time, are all requested before the first is added (in split order);
        // past the last split its values are requested again and not added
        const size_t zstride = (size_t)part_rows * part_cols;
#pragma unroll
        for (int it0 = 0; it0 < CHUNKS; it0 += 2) {
            float v[2][8];
#pragma unroll
            for (int c = 0; c < 2; c++)
#pragma unroll
                for (int e = 0; e < 8; e++) v[c][e] = 0.0f;
            const float* p0 = partial + (size_t)rowi * part_cols + at[it0];
            const float* p1 = partial + (size_t)rowi * part_cols + at[it0 + 1];
            for (uint32_t z0 = 0; z0 < splits; z0 += 3) {
                f32x4 lo[2][3], hi[2][3];
#pragma unroll
                for (uint32_t u = 0; u < 3; u++) {
                    const size_t zo = (size_t)(z0 + u < splits ? z0 + u : splits - 1) * zstride;
                    lo[0][u] = *reinterpret_cast<const f32x4*>(p0 + zo); hi[0][u] = *reinterpret_cast<const f32x4*>(p0 + zo + 4);
                    lo[1][u] = *reinterpret_cast<const f32x4*>(p1 + zo); hi[1][u] = *reinterpret_cast<const f32x4*>(p1 + zo + 4);
                }
                // All of them before the first addition: left to itself the compiler puts a split's loads behind the additions of the one before.
                asm volatile("" : "+v"(lo[0][0]), "+v"(hi[0][0]), "+v"(lo[1][0]), "+v"(hi[1][0]), "+v"(lo[0][1]), "+v"(hi[0][1]), "+v"(lo[1][1]), "+v"(hi[1][1]), "+v"(lo[0][2]),
                             "+v"(hi[0][2]), "+v"(lo[1][2]), "+v"(hi[1][2]));
#pragma unroll
                for (uint32_t u = 0; u < 3; u++) {
                    const bool in = z0 + u < splits;
#pragma unroll
                    for (int c = 0; c < 2; c++)
#pragma unroll
                        for (int e = 0; e < 8; e++) v[c][e] = in ? v[c][e] + (e < 4 ? lo : hi)[c][u][e & 3] : v[c][e];
                }
            }
#pragma unroll
            for (int c = 0; c < 2; c++)
                x[it0 + c] = make_uint4((uint32_t)lh_f2h(v[c][0]) | ((uint32_t)lh_f2h(v[c][1]) << 16), (uint32_t)lh_f2h(v[c][2]) | ((uint32_t)lh_f2h(v[c][3]) << 16),
                                        (uint32_t)lh_f2h(v[c][4]) | ((uint32_t)lh_f2h(v[c][5]) << 16), (uint32_t)lh_f2h(v[c][6]) | ((uint32_t)lh_f2h(v[c][7]) << 16));
        }
    } else {
#pragma unroll
        for (int it = 0; it < CHUNKS; it++) x[it] = *reinterpret_cast<const uint4*>(a.in + row + at[it]);
    }
    float s = 0.0f;
#pragma unroll
    for (int it = 0; it < CHUNKS; it++) {
        float t = s;
        rms_sumsq8(x[it], t);
        s = has[it] ? t : s;
    }
    const float rms = rsqrtf(block_sum(s, scratch, threads) / (float)dim + a.eps);
    float s2 = 0.0f;
#pragma unroll
    for (int it = 0; it < CHUNKS; it++) {
        o[it] = rms_apply8<ADD>(x[it], gw[it], ADD ? rr[it] : x[it], rms, 0u, 1.0f);
        if (a.apply_scale) o[it] = scale8(o[it], a.scale);
        float t = s2;
        rms_sumsq8(o[it], t);
        s2 = has[it] ? t : s2;
        if (has[it]) *reinterpret_cast<uint4*>(a.out + row + at[it]) = o[it];
    }
    if (nw2 == nullptr) return;
    const float rms2 = rsqrtf(block_sum(s2, scratch, threads) / (float)dim + a.eps);
#pragma unroll
    for (int it = 0; it < CHUNKS; it++)
        if (has[it]) *reinterpret_cast<uint4*>(a.out2 + row + at[it]) = rms_apply8<false>(o[it], gw2[it], o[it], rms2, 0u, 1.0f);
}

}  // namespace

bool lh_norm_fused_supported(uint32_t dim) { return (dim & 7) == 0 && dim <= 8192; }

void lh_launch_norm_fused(hipStream_t stream, const LhNormFused& a) {
    // the thread count launch_rms_norm picks for 16-byte accesses: the partial sums of the squares add up in the same order
    const uint32_t threads = a.dim >= 2048 ? 256u : (a.dim >= 1024 ? 128u : 64u);
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(a.rows), dim3(threads), 0, stream, a.w, a.res, a.w2, a.partial, a.dim, a.splits, a.part_rows, a.part_cols, threads, a);
    };
    const auto by_rows = [&](auto chunks) {
        constexpr int C = decltype(chunks)::value;
        if (a.partial) launch(a.res ? rms_norm_fused_kernel<true, true, C> : rms_norm_fused_kernel<true, false, C>);
        else launch(a.res ? rms_norm_fused_kernel<false, true, C> : rms_norm_fused_kernel<false, false, C>);
    };
    if (a.dim <= 16 * threads) by_rows(std::integral_constant<int, 2>{});
    else by_rows(std::integral_constant<int, 4>{});
}
