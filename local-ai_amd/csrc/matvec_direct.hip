// TQ2_0 and Q4_0 matvec (M = 1) for the products of one token: f16 out and in (or f32 in before a rotation), the vector in registers, no
// quantised activations.
//
// Same contract as matvec_tq2_mfma.hip and matvec_quant.hip (stands in for shaders/matvec_quant.metal:65-312).  A decoder's single
// products are a few megabytes: what bounds them is the length of the chain from the launch to the last row, not bytes or
// arithmetic.  The other forms have 16-bit limbs of the vector, tables and an LDS image of the weights in that chain; here a wave has its
// weights on their way before the vector is finished, and multiplies them as they arrive:
//   * 32 lanes take a row of up to 2048 columns, so a wave takes two rows at a time.  TQ2_0: lane l the quarter l % 4 of block l / 4 as one
//     16-byte load of codes, and the block's scale; Q4_0: the two blocks 2 l and 2 l + 1, 36 bytes.  Longer rows go to several waves,
//     whose sums meet in LDS.
//   * the vector after its prologue consists of f16 values, and a code less its zero point is exact in f16 too: v_dot2_f32_f16
//     multiplies them exactly (subnormal values included) and adds in f32; it truncates, so its sums stay short (four products).
// (Per launch in a token, weights cold: TQ2_0 2 x 6144 x 1536 behind the norms of a layer's end 10.2 us in the matrix-core form, 7.8 here;
// 1536 x 6144 behind GeGLU 12.2 and 6.2, 1536 x 12288 14.2 and 7.8.  Q4_0, against the form with v_dot4, one launch after the other: 2048 x 2048
// 5.0 and 3.8, 2 x 6144 x 1536 behind a norm 8.0 and 6.8, 1536 x 12288 behind GeGLU 14.3 and 7.8.)
#include "common.hpp"
#include "xquant.hpp"
#include <algorithm>

namespace {

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
template <class A>
__device__ __forceinline__ float lh_dot2h(A a, uint32_t b, float c) {
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, a), __builtin_bit_cast(f16x2, b), c, false);
}

struct DirectArgs {
    const uint8_t* m[8];       // `count` matrices of [rows][K / 256] blocks of 66 bytes or [rows][K / 32] of 18, all for the one vector
    uint16_t* y[8];
    const void* x;             // f16; before a rotation f32
    uint32_t count, rows, K;
    uint32_t batch, xstride, ystride;   // vectors, and bytes between them and between their outputs (several: one matrix, no prologue)
    XPrologue pro;
};

// A workgroup of ng x teams waves, ng = ceil(K / 2048): wave w takes the block group w % ng of the row pairs of team w / ng.
// NR: rounds of eight elements per thread that cover the vector.  V: vectors V blockIdx.y .. of a batch that the workgroup multiplies each
// code with once it is apart (the last ones may repeat the last vector); what a vector gives does not depend on V.
template <int FMT, int KIND, int NR, int MAXT, int V>
__global__ __launch_bounds__(MAXT) void matvec_direct_kernel(const DirectArgs a) {
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nthreads = blockDim.x;
    const uint32_t ng = (a.K + 2047) >> 11, teams = (nthreads >> 6) / ng, team = wave / ng, grp = wave - team * ng;
    uint4* const xs = reinterpret_cast<uint4*>(lds);                                   // [V][ng][8 chunks of 8 elements][32 lanes]
    float* const parts = reinterpret_cast<float*>(lds + (size_t)V * ng * 4096);         // [V][waves][64]
    float* const sums = parts + V * (nthreads >> 6) * 64;                               // [2][16]

    // ---- the vector, requested ahead of the weights: loads return in order
    static_assert(V == 1 || KIND == kXProNone, "a batch of vectors has no prologue");
    uint4 va[V * NR], vb[NR];
    [[maybe_unused]] uint4 vr[NR], vg[NR];
    [[maybe_unused]] float4 sa[NR], sb[NR];
    const uint32_t v0 = blockIdx.y * V;
#pragma unroll
    for (int i = 0; i < NR; i++) {
        const uint32_t e = min((i * nthreads + tid) * 8, a.K - 8);
        if constexpr (KIND == kXProRotate) {
            const float *x = static_cast<const float*>(a.x) + e, *s = a.pro.signs + (e & (a.pro.head_dim - 1));
            va[i] = *reinterpret_cast<const uint4*>(x);
            vb[i] = *reinterpret_cast<const uint4*>(x + 4);
            sa[i] = *reinterpret_cast<const float4*>(s);
            sb[i] = *reinterpret_cast<const float4*>(s + 4);
        } else
#pragma unroll
            for (int j = 0; j < V; j++)
                va[j * NR + i] = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(static_cast<const char*>(a.x) + (size_t)min(v0 + j, a.batch - 1) * a.xstride) + e);
        if constexpr (KIND == kXProRmsNorm || KIND == kXProGeluMul) vb[i] = *reinterpret_cast<const uint4*>(a.pro.aux + e);
        if constexpr (KIND == kXProRmsNorm) {
            const uint16_t* const xh = static_cast<const uint16_t*>(a.x);
            vr[i] = *reinterpret_cast<const uint4*>((a.pro.res ? a.pro.res : xh) + e);
            vg[i] = *reinterpret_cast<const uint4*>((a.pro.aux2 ? a.pro.aux2 : xh) + e);
        }
    }

    // ---- the weights of the first rows
    const uint32_t pairs = (a.rows + 1) >> 1, total = a.count * pairs;
    auto problem = [&](uint32_t q) { return a.count == 1 ? 0u : a.count == 2 ? (q >= pairs ? 1u : 0u) : q / pairs; };
    const uint32_t first = blockIdx.x * teams + team, step = gridDim.x * teams, count = first < total ? (total - first - 1) / step + 1 : 0u;
    const uint32_t half = lane >> 5, l = lane & 31, unit = min(32 * grp + l, (a.K >> 6) - 1);      // the lane's 64 weights of a row
    const uint32_t row_bytes = FMT == LH_TQ2_0 ? (a.K >> 8) * 66 : (a.K >> 5) * 18;
    const uint32_t code_off = FMT == LH_TQ2_0 ? (unit >> 2) * 66 + 16 * (unit & 3) : unit * 36, scale_off = (unit >> 2) * 66 + 64;
    struct Pair { u32x4_t w, w1; uint32_t d; } v[4];          // Q4_0: nine words
    auto issue = [&](Pair& p, uint32_t i) {
        const uint32_t q = min(first + i * step, total - 1), pr = problem(q), row = min(2 * (q - pr * pairs) + half, a.rows - 1);
        const uint8_t* src = (a.count <= 2 ? (pr ? a.m[1] : a.m[0]) : a.m[pr]) + (size_t)row * row_bytes;
        typedef u32x4_t __attribute__((aligned(2))) u32x4_ua;   // (Q4_0: four bytes)
        p.w = __builtin_nontemporal_load(reinterpret_cast<const u32x4_ua*>(src + code_off));
        if constexpr (FMT == LH_TQ2_0) p.d = *reinterpret_cast<const uint16_t*>(src + scale_off);
        else {
            p.w1 = __builtin_nontemporal_load(reinterpret_cast<const u32x4_ua*>(src + code_off + 16));
            p.d = *reinterpret_cast<const uint32_t*>(src + code_off + 32);
        }
    };
    lh_first_rows(v, max(count, 1u), issue);

    // ---- the prologue: f16 values in LDS, a lane's eight chunks of a block group in the order in which it reads them
    auto total_of = [&](float s, float* sums) {
        s = lh_group_sum(s, 64);
        if (lane == 0) sums[wave] = s;
        lh_lds_barrier();
        float t = 0.0f;
#pragma unroll
        for (uint32_t w = 0; w < MAXT / 64; w++) t += w < nthreads >> 6 ? sums[w] : 0.0f;
        return t;
    };
    auto square = [](const uint4 v) {
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float lo = lh_h2f((uint16_t)(w[j] & 0xFFFF)), hi = lh_h2f((uint16_t)(w[j] >> 16));
            s += lo * lo;
            s += hi * hi;
        }
        return s;
    };
    [[maybe_unused]] float rms = 1.0f, rms2 = 1.0f;
    if constexpr (KIND == kXProRmsNorm) {
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < NR; i++) s += (i * nthreads + tid) * 8 < a.K ? square(va[i]) : 0.0f;
        rms = rsqrtf(total_of(s, sums) / (float)a.K + a.pro.eps);
        s = 0.0f;
#pragma unroll
        for (int i = 0; i < NR; i++) {
            const uint32_t e = (i * nthreads + tid) * 8;
            uint32_t n[4];
            xpro_norm_add8_regs(va[i], vb[i], vr[i], a.pro, rms, n);
            va[i] = make_uint4(n[0], n[1], n[2], n[3]);
            s += e < a.K ? square(va[i]) : 0.0f;
            if (e < a.K && a.pro.store && blockIdx.x == 0) *reinterpret_cast<uint4*>(a.pro.store + e) = va[i];
        }
        if (a.pro.aux2) rms2 = rsqrtf(total_of(s, sums + 16) / (float)a.K + a.pro.eps);
    }
#pragma unroll
    for (int p = 0; p < V * NR; p++) {
        const int i = p % NR;
        const uint32_t e = (i * nthreads + tid) * 8;
        const bool in = e < a.K;
        uint32_t w[4] = {va[p].x, va[p].y, va[p].z, va[p].w};
        if constexpr (KIND == kXProRmsNorm) {
            if (a.pro.aux2) {
                const uint32_t g[4] = {vg[i].x, vg[i].y, vg[i].z, vg[i].w};
#pragma unroll
                for (int j = 0; j < 4; j++)
                    w[j] = (uint32_t)lh_f2h_exact(lh_norm_product(lh_h2f((uint16_t)(w[j] & 0xFFFF)), rms2, lh_h2f((uint16_t)(g[j] & 0xFFFF)))) |
                           (uint32_t)lh_f2h_exact(lh_norm_product(lh_h2f((uint16_t)(w[j] >> 16)), rms2, lh_h2f((uint16_t)(g[j] >> 16)))) << 16;
            }
        }
        if constexpr (KIND == kXProGeluMul) {
            const uint32_t b[4] = {vb[i].x, vb[i].y, vb[i].z, vb[i].w};
#pragma unroll
            for (int j = 0; j < 4; j++)
                w[j] = (uint32_t)lh_gelu_mul_h((uint16_t)(w[j] & 0xFFFF), (uint16_t)(b[j] & 0xFFFF)) |
                       (uint32_t)lh_gelu_mul_h((uint16_t)(w[j] >> 16), (uint16_t)(b[j] >> 16)) << 16;
        }
        if constexpr (KIND == kXProRotate) {
            float t[8] = {__uint_as_float(va[i].x), __uint_as_float(va[i].y), __uint_as_float(va[i].z), __uint_as_float(va[i].w),
                          __uint_as_float(vb[i].x), __uint_as_float(vb[i].y), __uint_as_float(vb[i].z), __uint_as_float(vb[i].w)};
            xpro_rotate8_regs(t, a.pro, sa[i], sb[i]);
#pragma unroll
            for (int j = 0; j < 4; j++) w[j] = (uint32_t)lh_f2h(t[2 * j]) | (uint32_t)lh_f2h(t[2 * j + 1]) << 16;
        }
        // TQ2_0: element e of a block is in half e / 128, field e / 32 % 4, byte 16 (e / 16 % 2) + e % 16: lane 4 b + 2 half + e / 16 % 2, chunk
        // 2 field + e / 8 % 2.  Q4_0: chunk e / 8 % 8 of lane e / 64, the elements in the order 0 2 1 3 in which the nibbles come apart.
        if (e < ng * 2048) {
            const uint32_t chunk = FMT == LH_TQ2_0 ? 2 * ((e >> 5) & 3) + ((e >> 3) & 1) : (e >> 3) & 7;
            const uint32_t to = FMT == LH_TQ2_0 ? 4 * ((e >> 8) & 7) + 2 * ((e >> 7) & 1) + ((e >> 4) & 1) : (e >> 6) & 31;
            if constexpr (FMT == LH_Q4_0)
#pragma unroll
                for (int j = 0; j < 4; j += 2) {
                    const uint32_t lo = w[j], hi = w[j + 1];
                    w[j] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
                    w[j + 1] = __builtin_amdgcn_perm(hi, lo, 0x07060302u);
                }
            xs[((p / NR * ng + (e >> 11)) * 8 + chunk) * 32 + to] = in ? make_uint4(w[0], w[1], w[2], w[3]) : make_uint4(0u, 0u, 0u, 0u);
        }
    }
    lh_lds_barrier();
    uint32_t x[V][8][4];                                      // the lane's eight chunks
#pragma unroll
    for (int j = 0; j < V; j++)
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const uint4 t = xs[((j * ng + grp) * 8 + c) * 32 + l];
            x[j][c][0] = t.x; x[j][c][1] = t.y; x[j][c][2] = t.z; x[j][c][3] = t.w;
        }

    float mine[V];                                            // lane 32 h + i: row h of the wave's pair i (32 of them at most)
#pragma unroll
    for (int j = 0; j < V; j++) mine[j] = 0.0f;
    lh_walk_rows(v, count, issue, [&](const Pair& p, uint32_t i) {
        float part[V];
        if constexpr (FMT == LH_TQ2_0) {
            float acc[V][4];
#pragma unroll
            for (int j = 0; j < V; j++)
#pragma unroll
                for (int f = 0; f < 4; f++) acc[j][f] = 0.0f;
#pragma unroll
            for (int m = 0; m < 4; m++)
#pragma unroll
                for (int f = 0; f < 4; f++) {
                    // the high bytes of f16(code - 1), the low ones are zero: four at a time from a table, then apart
                    const uint32_t hi = __builtin_amdgcn_perm(0u, 0x403C00BCu, (p.w[m] >> (2 * f)) & 0x03030303u);
                    const uint32_t c0 = __builtin_amdgcn_perm(0u, hi, 0x010C000Cu), c1 = __builtin_amdgcn_perm(0u, hi, 0x030C020Cu);
#pragma unroll
                    for (int j = 0; j < V; j++) {
                        const uint32_t* xc = &x[j][2 * f + (m >> 1)][2 * (m & 1)];
                        acc[j][f] += lh_dot2h(c0, xc[0], lh_dot2h(c1, xc[1], 0.0f));
                    }
                }
#pragma unroll
            for (int j = 0; j < V; j++) {
                part[j] = ((acc[j][0] + acc[j][1]) + (acc[j][2] + acc[j][3])) * lh_h2f((uint16_t)p.d);
                asm volatile("" : "+v"(part[j]));             // rounded here, not in an addition of the sum over the lanes: in every variant the same
            }
        } else {
            // scale, 4 words of codes; twice: the first block's codes lie two bytes into a word
            const uint32_t w[9] = {p.w[0], p.w[1], p.w[2], p.w[3], p.w1[0], p.w1[1], p.w1[2], p.w1[3], p.d};
#pragma unroll
            for (int j = 0; j < V; j++) part[j] = 0.0f;
#pragma unroll
            for (int b = 0; b < 2; b++) {
                float acc[V][2];
#pragma unroll
                for (int j = 0; j < V; j++) acc[j][0] = acc[j][1] = 0.0f;
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    const uint32_t c = b ? w[5 + m] : __builtin_amdgcn_alignbit(w[m + 1], w[m], 16), c8 = c >> 8;
                    // f16(1024 + nibble) less 1032, f16(1024 + 16 nibble) / 16 less 72: both exact
                    const f16x2 one = {(_Float16)1.0f, (_Float16)1.0f}, sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f}, z = {(_Float16)-1032.0f, (_Float16)-1032.0f},
                                z16 = {(_Float16)-72.0f, (_Float16)-72.0f};
                    const f16x2 lo0 = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, (c & 0x000F000Fu) | 0x64006400u), one, z);
                    const f16x2 lo1 = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, (c8 & 0x000F000Fu) | 0x64006400u), one, z);
                    const f16x2 hi0 = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, (c & 0x00F000F0u) | 0x64006400u), sixteenth, z16);
                    const f16x2 hi1 = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, (c8 & 0x00F000F0u) | 0x64006400u), sixteenth, z16);
#pragma unroll
                    for (int j = 0; j < V; j++) {
                        const uint32_t *xl = &x[j][4 * b + (m >> 1)][2 * (m & 1)], *xh = &x[j][4 * b + 2 + (m >> 1)][2 * (m & 1)];
                        acc[j][0] += lh_dot2h(lo0, xl[0], lh_dot2h(lo1, xl[1], 0.0f));
                        acc[j][1] += lh_dot2h(hi0, xh[0], lh_dot2h(hi1, xh[1], 0.0f));
                    }
                }
#pragma unroll
                for (int j = 0; j < V; j++) part[j] = __builtin_fmaf(acc[j][0] + acc[j][1], lh_h2f((uint16_t)(b ? w[4] >> 16 : w[0] & 0xFFFFu)), part[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < V; j++) {
            const float sum = lh_group_sum(part[j], 32);
            mine[j] = i == l ? sum : mine[j];
        }
    });
    const uint32_t waves = nthreads >> 6;
    if (ng > 1) {
#pragma unroll
        for (int j = 0; j < V; j++) parts[(j * waves + wave) * 64 + lane] = mine[j];
        lh_lds_barrier();
        if (grp != 0) return;
#pragma unroll
        for (int j = 0; j < V; j++)
            for (uint32_t g = 1; g < ng; g++) mine[j] += parts[(j * waves + wave + g) * 64 + lane];
    }
    if (l < count) {
        const uint32_t q = first + l * step, pr = problem(q), row = 2 * (q - pr * pairs) + half;
        if (row < a.rows)
#pragma unroll
            for (int j = 0; j < V; j++)
                if (v0 + j < a.batch) reinterpret_cast<uint16_t*>(reinterpret_cast<char*>(a.y[pr]) + (size_t)(v0 + j) * a.ystride)[row] = lh_f2h(mine[j]);
    }
}

}  // namespace

int lh_launch_matvec_direct(lh_context* ctx, lh_quant fmt, uint32_t count, const void* const* matrices, const void* vector, void* const* outputs, uint32_t rows,
                                uint32_t K, const XPrologue& pro, uint32_t batch, uint32_t xstride, uint32_t ystride) {
    const uint32_t ng = (K + 2047) / 2048;
    if (count > 8 || ng > 6 || (batch > 1 && (count > 1 || pro.kind != kXProNone))) return -1;
    const uint32_t waves = ng == 1 || ng == 2 || ng == 4 ? 8 : 2 * ng, teams = waves / ng, rounds = (ng * 2048 + waves * 512 - 1) / (waves * 512);   // rounds: 1 or 2
    // Beyond 8 pairs of rows per wave of a workgroup per CU (16 where a row takes several waves) the unpacking is what takes the time, and
    // the matrix cores do the rest of the work for nothing: 65536 x 1536 (16 per wave) 13.1 us against 11.2 there, 32768 x 2048 (8) 8.3
    // against 8.7; 16384 x 12288 (16) 19.1 against 22.2.  The line does not depend on the batch: what a vector gives alone it gives in one.
    const uint64_t total = (uint64_t)((rows + 1) / 2) * count, slots = (uint64_t)ctx->cu_count * teams;
    if (total > slots * (ng == 1 ? 8 : 16)) return -1;
    // Vectors of a batch that share the unpacked codes.  Up to a pair of rows per wave (three where a row takes several) each vector has
    // workgroups of its own, then two share one, from nine on four, where there are 256 registers for them.  Q4_0, in microseconds with 1, 2 and 4, and in
    // the form with v_dot4: 8 x 256 x 1536 3.6, 4.0, 5.2, 4.6; 3 x 1536 x 2048 5.0, 4.3, 5.3, 5.9; 4 x 8960 x 1536 9.7, 8.1, 8.8, 10.5;
    // 8 x 24576 x 1536 46, 27, 23, 27.
    const uint64_t load = batch * total;
    const uint32_t v = batch == 1 || load <= slots * (ng == 1 ? 1 : 3) ? 1 : batch > 2 && waves <= 8 && load >= slots * 9 ? 4 : 2;
    const uint32_t groups = (batch + v - 1) / v;
    // A workgroup per CU, and a wave's results fit its half of the lanes.
    const uint64_t fill = std::max<uint64_t>({(uint64_t)ctx->cu_count / groups, 1, (total + (uint64_t)teams * 32 - 1) / ((uint64_t)teams * 32)});
    const dim3 grid((uint32_t)std::min<uint64_t>((total + teams - 1) / teams, fill), groups);
    DirectArgs a{{}, {}, vector, count, rows, K, batch, xstride, ystride, pro};
    for (uint32_t i = 0; i < count; i++) { a.m[i] = (const uint8_t*)matrices[i]; a.y[i] = (uint16_t*)outputs[i]; }
    const size_t lds = (size_t)v * ng * 4096 + ((size_t)v * waves * 64 + 32) * 4;
    int r = LH_OK;
#define LH_DIRECT_V(FMT, KIND, NR, MAXT, V)                                                                                                              \
    do {                                                                                                                                                 \
        if (lds > 65536) r = lh_raise_dynamic_lds(ctx, (const void*)matvec_direct_kernel<FMT, KIND, NR, MAXT, V>, lds, "matvec_quant");                   \
        if (r == LH_OK) hipLaunchKernelGGL((matvec_direct_kernel<FMT, KIND, NR, MAXT, V>), grid, dim3(64 * waves), lds, ctx->stream, a);                 \
    } while (0)
#define LH_DIRECT(FMT, KIND, NR)                                         \
    do {                                                                 \
        if (v == 4) LH_DIRECT_V(FMT, kXProNone, NR, 512, 4);             \
        else if (v == 2 && waves <= 8) LH_DIRECT_V(FMT, kXProNone, NR, 512, 2); \
        else if (v == 2) LH_DIRECT_V(FMT, kXProNone, NR, 768, 2);        \
        else if (waves <= 8) LH_DIRECT_V(FMT, KIND, NR, 512, 1);         \
        else LH_DIRECT_V(FMT, KIND, NR, 768, 1);                         \
    } while (0)
#define LH_DIRECT_KIND(FMT, KIND) do { if (rounds == 1) LH_DIRECT(FMT, KIND, 1); else LH_DIRECT(FMT, KIND, 2); } while (0)
#define LH_DIRECT_FMT(FMT)                                                    \
    do {                                                                      \
        if (pro.kind == kXProRmsNorm) LH_DIRECT_KIND(FMT, kXProRmsNorm);      \
        else if (pro.kind == kXProGeluMul) LH_DIRECT_KIND(FMT, kXProGeluMul); \
        else if (pro.kind == kXProRotate) LH_DIRECT_KIND(FMT, kXProRotate);   \
        else LH_DIRECT_KIND(FMT, kXProNone);                                  \
    } while (0)
    if (fmt == LH_TQ2_0) LH_DIRECT_FMT(LH_TQ2_0);
    else LH_DIRECT_FMT(LH_Q4_0);
#undef LH_DIRECT_FMT
#undef LH_DIRECT_KIND
#undef LH_DIRECT
    return r != LH_OK ? r : lh_check_launch(fmt == LH_TQ2_0 ? "matvec_tq2_0" : "matvec_q4_0");
}
