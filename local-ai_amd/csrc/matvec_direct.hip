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
// (Per launch in a token, weights cold: TQ2_0 2 x 6144 x 1536 behind the norms of a layer's end 10.2 us in the matrix-core form; with 2 x 12288 x 1536
// 8.5 on average in this one at first, and 7.2 since the first loads' arguments arrive with the wave, all waves share the prologue and the vector is requested ahead
// of the weights; 1536 x 6144 behind GeGLU 12.2, 6.1 and now 4.5, 1536 x 12288 14.2, 7.5 and 5.7, that product being formed by the launch in front.  Q4_0,
// against the form with v_dot4, one launch after the other: 2048 x 2048 5.0 and 3.6, 2 x 6144 x 1536 behind a norm 8.0 and 6.8; in a token 1536 x 2048
// behind a rotation 5.4 and now 4.0.)
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
// Two codes of a word, where `mask` has them in the low bytes of its halves, less their zero point (`zero`, at the codes' place): exact, as the f16 value
// 1024 + code less 1024 + zero.  `base`: 1024 twice, in a vector register, so that taking and setting the bits is one instruction.  A word of sixteen TQ2_0
// codes takes 37 instructions with its products.  (Codes as they are, the vector's sum taken off in the end: 36, but the two sums nearly cancel, with 2 to 4 times
// the f32 error for vectors of one sign or with a large element, and weights of zero did not give zero; byte permutes: 39.  46 shapes of one f16 vector: 4 % longer
// with the sums.)
__device__ __forceinline__ f16x2 code_values(uint32_t word, uint32_t mask, uint32_t base, uint32_t zero) {
    const _Float16 less = (_Float16)(float)(1024u + zero);
    return __builtin_bit_cast(f16x2, (word & mask) | base) - (f16x2){less, less};
}

struct DirectArgs {
    const uint8_t* m[8];       // `count` matrices of [rows][K / 256] blocks of 66 bytes or [rows][K / 32] of 18, all for the one vector
    uint16_t* y[8];
    uint32_t count, pairs, total;       // pairs of rows of a matrix, of all of them (kGated: pairs are a row of each)
    uint32_t share, more;               // pairs of a team: `share`, and one more for the first `more`
    uint32_t batch, xstride, ystride;   // vectors, and bytes between them and between their outputs (several: one matrix, no prologue)
    uint16_t* store;                    // the prologue's other words, see XPrologue
    float eps, scale;
    uint32_t tail, head_dim;
    uint32_t has_res, has_next;         // whether there are a residual and a second norm
    const uint16_t* factor;             // kFactor: f16[rows]
};

// Waves of a workgroup for rows of NG groups of 2048 columns, and elements of the vector that a thread takes at a time: four where that
// covers the vector, so that all waves share the prologue (eight for a rotation, whose first three stages pair a thread's own).
constexpr int direct_waves(int ng) { return ng == 1 || ng == 2 || ng == 4 ? 8 : 2 * ng; }
constexpr int direct_elements(int ng, int kind) { return ng == 1 && kind != (int)kXProRotate ? 4 : 8; }

// The matrices of a launch: one; several, each with results of its own; or a gate and an up projection whose rows of one index are the two
// halves of a wave, which leaves gelu(gate) * up of the two f16 results; or one whose results leave as gelu(result) * factor.  (The product
// behind them would make the same of them in its prologue, but each of its workgroups again: a quantized token of ten
// layers 659 us with those prologues, 640 without.  Both launches, with the prologue and without, TQ2_0: two of 1024 rows, four to six groups of columns,
// 8192 12.6 us and 10.9, 10240 14.4 and 12.6, 12288 15.1 and 13.2; one of 512 rows 11.0 and 9.7, 12.4 and 11.1, 12.9 and 11.6; Q4_0 alike, 164 shapes 0.84.)
enum : int { kOne = 0, kSeveral = 1, kGated = 2, kFactor = 3 };

template <int E> struct Elements { uint32_t w[E / 2]; };
template <int E>
__device__ __forceinline__ Elements<E> load_elements(const uint16_t* p) {
    Elements<E> r;
    if constexpr (E == 8) { const uint4 t = *reinterpret_cast<const uint4*>(p); r.w[0] = t.x; r.w[1] = t.y; r.w[2] = t.z; r.w[3] = t.w; }
    else { const uint2 t = *reinterpret_cast<const uint2*>(p); r.w[0] = t.x; r.w[1] = t.y; }
    return r;
}

// A use of what a load brings, without an instruction.
template <int E>
__device__ __forceinline__ void keep(const Elements<E>& v) {
#pragma unroll
    for (int j = 0; j < E / 2; j++) asm volatile("" :: "v"(v.w[j]));
}
__device__ __forceinline__ void keep(const float4& v) { asm volatile("" :: "v"(v.x), "v"(v.y), "v"(v.z), "v"(v.w)); }

// A workgroup of TEAMS x NG waves: wave w takes the block group w % NG of the row pairs of team w / NG.  V: vectors V blockIdx.y .. of a
// batch that the workgroup multiplies each code with once it is apart (the last ones may repeat the last vector); what a vector gives does
// not depend on V.
// What the first loads need stands in front, one by one: such arguments arrive in registers with the wave (the Makefile asks for it), where
// the first word of a structure is 0.28 us away, in host memory.
// `second`: the norm weight, the second factor, or the signs; `res`, `aux2`: see XPrologue (the vector itself where there are none).
template <int FMT, int KIND, int NG, int V, int M>
__global__ __launch_bounds__(64 * direct_waves(NG)) void matvec_direct_kernel(const void* vector, const uint16_t* second, const uint16_t* res, const uint16_t* aux2,
                                                                              const uint8_t* m0, uint32_t K, uint32_t rows, uint32_t step, const DirectArgs a) {
    constexpr int WAVES = direct_waves(NG), TEAMS = WAVES / NG, NT = 64 * WAVES, E = direct_elements(NG, KIND), NR = (NG * 2048 + NT * E - 1) / (NT * E), W = E / 2;
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t team = wave / NG, grp = wave - team * NG;
    uint2* const xs = reinterpret_cast<uint2*>(lds);                                    // [V][NG][8 chunks of 8 elements][32 lanes][2]
    float* const parts = reinterpret_cast<float*>(lds + (size_t)V * NG * 4096);         // [V][waves][64]
    float* const sums = parts + V * WAVES * 64;                                         // [2][16]

    // ---- the vector, requested ahead of the weights: loads return in order
    static_assert(V == 1 || KIND == kXProNone, "a batch of vectors has no prologue");
    Elements<E> va[V * NR];
    [[maybe_unused]] Elements<E> vb[NR], vr[NR], vg[NR];
    [[maybe_unused]] float4 fa[NR], fb[NR], sa[NR], sb[NR];
    const uint32_t v0 = blockIdx.y * V;
#pragma unroll
    for (int i = 0; i < NR; i++) {
        const uint32_t e = min((i * NT + tid) * E, K - E);
        if constexpr (KIND == kXProRotate) {
            const float *x = static_cast<const float*>(vector) + e, *s = reinterpret_cast<const float*>(second) + (e & (a.head_dim - 1));
            fa[i] = *reinterpret_cast<const float4*>(x);
            fb[i] = *reinterpret_cast<const float4*>(x + 4);
            sa[i] = *reinterpret_cast<const float4*>(s);
            sb[i] = *reinterpret_cast<const float4*>(s + 4);
        } else
#pragma unroll
            for (int j = 0; j < V; j++) {
                const char* x = static_cast<const char*>(vector);
                if constexpr (KIND == kXProNone) x += (size_t)min(v0 + j, a.batch - 1) * a.xstride;
                va[j * NR + i] = load_elements<E>(reinterpret_cast<const uint16_t*>(x) + e);
            }
        if constexpr (KIND == kXProRmsNorm || KIND == kXProGeluMul) vb[i] = load_elements<E>(second + e);
        if constexpr (KIND == kXProRmsNorm) {
            vr[i] = load_elements<E>(res + e);
            vg[i] = load_elements<E>(aux2 + e);
        }
    }

    // ---- the weights of the first rows
    const uint32_t pairs = a.pairs;
    auto problem = [&](uint32_t q) { return M != kSeveral ? 0u : a.count == 2 ? (q >= pairs ? 1u : 0u) : q / pairs; };
    const uint32_t first = blockIdx.x * TEAMS + team, count = a.share + (first < a.more ? 1u : 0u);
    const uint32_t half = lane >> 5, l = lane & 31, unit = min(32 * grp + l, (K >> 6) - 1);      // the lane's 64 weights of a row
    const uint32_t row_bytes = FMT == LH_TQ2_0 ? (K >> 8) * 66 : (K >> 5) * 18;
    const uint32_t code_off = FMT == LH_TQ2_0 ? (unit >> 2) * 66 + 16 * (unit & 3) : unit * 36, scale_off = (unit >> 2) * 66 + 64;
    struct Pair { u32x4_t w, w1; uint32_t d; } v[4];          // Q4_0: nine words
    auto issue = [&](Pair& p, uint32_t i) {
        const uint32_t q = min(first + i * step, a.total - 1), pr = problem(q), row = M == kGated ? q : min(2 * (q - pr * pairs) + half, rows - 1);
        const uint8_t* src = m0;
        if constexpr (M == kGated) src = half ? a.m[1] : m0;
        else if constexpr (M == kSeveral) if (pr) src = a.m[pr];
        src += (size_t)row * row_bytes;
        typedef u32x4_t __attribute__((aligned(2))) u32x4_ua;   // (Q4_0: four bytes)
        p.w = __builtin_nontemporal_load(reinterpret_cast<const u32x4_ua*>(src + code_off));
        if constexpr (FMT == LH_TQ2_0) p.d = *reinterpret_cast<const uint16_t*>(src + scale_off);
        else {
            p.w1 = __builtin_nontemporal_load(reinterpret_cast<const u32x4_ua*>(src + code_off + 16));
            p.d = *reinterpret_cast<const uint32_t*>(src + code_off + 32);
        }
    };
    [[maybe_unused]] uint16_t factor = 0;
    if constexpr (M == kFactor) factor = a.factor[min(2 * (first + l * step) + half, rows - 1)];
    lh_first_rows(v, max(count, 1u), issue);

    // ---- the prologue: f16 values in LDS, a lane's eight chunks of a block group in the order in which it reads them
    auto total_of = [&](float s, float* sums) {
        s = lh_group_sum(s, 64);
        if (lane == 0) sums[wave] = s;
        lh_lds_barrier();
        float t = 0.0f;
#pragma unroll
        for (int w = 0; w < WAVES; w++) t += sums[w];
        return t;
    };
    auto square = [](const Elements<E>& v) {
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < W; j++) {
            const float lo = lh_h2f((uint16_t)(v.w[j] & 0xFFFF)), hi = lh_h2f((uint16_t)(v.w[j] >> 16));
            s += lo * lo;
            s += hi * hi;
        }
        return s;
    };
    // (whether a wave has any of the vector's elements: those that have none leave their SIMD to the others)
    auto has = [&](int i) { return (i * NT + 64 * wave) * E < K; };
    [[maybe_unused]] float rms = 1.0f, rms2 = 1.0f;
    if constexpr (KIND == kXProRmsNorm) {
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < NR; i++) if (has(i)) s += (i * NT + tid) * E < K ? square(va[i]) : 0.0f;
        rms = rsqrtf(total_of(s, sums) / (float)K + a.eps);
        s = 0.0f;
#pragma unroll
        for (int i = 0; i < NR; i++) {
            if (!has(i)) continue;
            const uint32_t e = (i * NT + tid) * E;
#pragma unroll
            for (int j = 0; j < W; j++) {                     // the arithmetic of rms_norm_kernel<ADD>, its tail forms included
                float lo = lh_norm_product(lh_h2f((uint16_t)(va[i].w[j] & 0xFFFF)), rms, lh_h2f((uint16_t)(vb[i].w[j] & 0xFFFF)));
                float hi = lh_norm_product(lh_h2f((uint16_t)(va[i].w[j] >> 16)), rms, lh_h2f((uint16_t)(vb[i].w[j] >> 16)));
                if (a.has_res) {
                    const float rlo = lh_h2f((uint16_t)(vr[i].w[j] & 0xFFFF)), rhi = lh_h2f((uint16_t)(vr[i].w[j] >> 16));
                    if (a.tail) { lo = lh_norm_tail(lo, rlo, a.tail, a.scale); hi = lh_norm_tail(hi, rhi, a.tail, a.scale); }
                    else { lo += rlo; hi += rhi; }
                }
                va[i].w[j] = (uint32_t)lh_f2h_exact(lo) | ((uint32_t)lh_f2h_exact(hi) << 16);
            }
            s += e < K ? square(va[i]) : 0.0f;
            if (e < K && a.store && blockIdx.x == 0) {
                if constexpr (E == 8) *reinterpret_cast<uint4*>(a.store + e) = make_uint4(va[i].w[0], va[i].w[1], va[i].w[2], va[i].w[3]);
                else *reinterpret_cast<uint2*>(a.store + e) = make_uint2(va[i].w[0], va[i].w[1]);
            }
        }
        if (a.has_next) rms2 = rsqrtf(total_of(s, sums + 16) / (float)K + a.eps);
    }
#pragma unroll
    for (int p = 0; p < V * NR; p++) {
        const int i = p % NR;
        const uint32_t e = (i * NT + tid) * E;
        uint32_t w[W];
#pragma unroll
        for (int j = 0; j < W; j++) w[j] = 0u;
        if (has(i)) {
            if constexpr (KIND == kXProRotate) {
                float t[8] = {fa[i].x, fa[i].y, fa[i].z, fa[i].w, fb[i].x, fb[i].y, fb[i].z, fb[i].w};
                xpro_rotate8_regs<false>(t, a.head_dim, a.scale, sa[i], sb[i]);
#pragma unroll
                for (int j = 0; j < W; j++) w[j] = (uint32_t)lh_f2h(t[2 * j]) | (uint32_t)lh_f2h(t[2 * j + 1]) << 16;
            } else
#pragma unroll
                for (int j = 0; j < W; j++) {
                    w[j] = va[p].w[j];
                    const uint16_t lo = (uint16_t)(w[j] & 0xFFFF), hi = (uint16_t)(w[j] >> 16);
                    if constexpr (KIND == kXProRmsNorm) {
                        if (a.has_next)
                            w[j] = (uint32_t)lh_f2h_exact(lh_norm_product(lh_h2f(lo), rms2, lh_h2f((uint16_t)(vg[i].w[j] & 0xFFFF)))) |
                                   (uint32_t)lh_f2h_exact(lh_norm_product(lh_h2f(hi), rms2, lh_h2f((uint16_t)(vg[i].w[j] >> 16)))) << 16;
                    }
                    if constexpr (KIND == kXProGeluMul)
                        w[j] = (uint32_t)lh_gelu_mul_h(lo, (uint16_t)(vb[i].w[j] & 0xFFFF)) | (uint32_t)lh_gelu_mul_h(hi, (uint16_t)(vb[i].w[j] >> 16)) << 16;
                }
            if (e >= K)
#pragma unroll
                for (int j = 0; j < W; j++) w[j] = 0u;
        } else {                                              // (or the compiler would request them here, behind the weights)
            if constexpr (KIND == kXProRotate) { keep(fa[i]); keep(fb[i]); keep(sa[i]); keep(sb[i]); }
            else keep(va[p]);
            if constexpr (KIND == kXProGeluMul) keep(vb[i]);
        }
        // TQ2_0: element e of a block is in half e / 128, field e / 32 % 4, byte 16 (e / 16 % 2) + e % 16: lane 4 b + 2 half + e / 16 % 2, chunk
        // 2 field + e / 8 % 2.  Q4_0: chunk e / 8 % 8 of lane e / 64.  Four elements in the order 0 2 1 3 in which a word's codes come apart.
        if (e < NG * 2048) {
            const uint32_t chunk = FMT == LH_TQ2_0 ? 2 * ((e >> 5) & 3) + ((e >> 3) & 1) : (e >> 3) & 7;
            const uint32_t to = FMT == LH_TQ2_0 ? 4 * ((e >> 8) & 7) + 2 * ((e >> 7) & 1) + ((e >> 4) & 1) : (e >> 6) & 31;
#pragma unroll
            for (int j = 0; j < W; j += 2) {
                const uint32_t lo = w[j], hi = w[j + 1];
                w[j] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
                w[j + 1] = __builtin_amdgcn_perm(hi, lo, 0x07060302u);
            }
            uint2* const at = xs + ((((p / NR * NG + (e >> 11)) * 8 + chunk) * 32 + to) * 2);
            if constexpr (E == 8) *reinterpret_cast<uint4*>(at) = make_uint4(w[0], w[1], w[2], w[3]);
            else at[(e >> 2) & 1] = make_uint2(w[0], w[1]);
        }
    }
    lh_lds_barrier();
    uint32_t x[V][8][4];                                      // the lane's eight chunks
#pragma unroll
    for (int j = 0; j < V; j++)
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const uint4 t = *reinterpret_cast<const uint4*>(xs + (((j * NG + grp) * 8 + c) * 32 + l) * 2);
            x[j][c][0] = t.x; x[j][c][1] = t.y; x[j][c][2] = t.z; x[j][c][3] = t.w;
        }
    float mine[V];                                            // lane 32 h + i: row h of the wave's pair i (32 of them at most)
#pragma unroll
    for (int j = 0; j < V; j++) mine[j] = 0.0f;
    uint32_t base = 0x64006400u;
    asm("" : "+v"(base));
    lh_walk_rows(v, count, issue, [&](const Pair& p, uint32_t i) {
        float part[V];
        if constexpr (FMT == LH_TQ2_0) {
            float acc[V][4];
#pragma unroll
            for (int m = 0; m < 4; m++) {
                const uint32_t c = p.w[m], c8 = c >> 8;
#pragma unroll
                for (int f = 0; f < 4; f++) {
                    const uint32_t mask = 0x00030003u << (2 * f), zero = 1u << (2 * f);
                    const f16x2 even = code_values(c, mask, base, zero), odd = code_values(c8, mask, base, zero);      // bytes 0, 2 and 1, 3
#pragma unroll
                    for (int j = 0; j < V; j++) {
                        const uint32_t* xc = &x[j][2 * f + (m >> 1)][2 * (m & 1)];
                        const float four = lh_dot2h(even, xc[0], lh_dot2h(odd, xc[1], 0.0f));
                        acc[j][f] = m ? acc[j][f] + four : four;
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < V; j++) {
                part[j] = (__builtin_fmaf(acc[j][1], 0.25f, acc[j][0]) + __builtin_fmaf(acc[j][3], 0.015625f, acc[j][2] * 0.0625f)) * lh_h2f((uint16_t)p.d);
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
                for (int m = 0; m < 4; m++) {
                    const uint32_t c = b ? w[5 + m] : __builtin_amdgcn_alignbit(w[m + 1], w[m], 16), c8 = c >> 8;
                    const f16x2 lo0 = code_values(c, 0x000F000Fu, base, 8), lo1 = code_values(c8, 0x000F000Fu, base, 8);
                    const f16x2 hi0 = code_values(c, 0x00F000F0u, base, 128), hi1 = code_values(c8, 0x00F000F0u, base, 128);
#pragma unroll
                    for (int j = 0; j < V; j++) {
                        const uint32_t *xl = &x[j][4 * b + (m >> 1)][2 * (m & 1)], *xh = &x[j][4 * b + 2 + (m >> 1)][2 * (m & 1)];
                        const float lo = lh_dot2h(lo0, xl[0], lh_dot2h(lo1, xl[1], 0.0f)), hi = lh_dot2h(hi0, xh[0], lh_dot2h(hi1, xh[1], 0.0f));
                        acc[j][0] = m ? acc[j][0] + lo : lo;
                        acc[j][1] = m ? acc[j][1] + hi : hi;
                    }
                }
#pragma unroll
                for (int j = 0; j < V; j++)
                    part[j] = __builtin_fmaf(__builtin_fmaf(acc[j][1], 0.0625f, acc[j][0]), lh_h2f((uint16_t)(b ? w[4] >> 16 : w[0] & 0xFFFFu)), part[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < V; j++) {
            const float sum = lh_group_sum(part[j], 32);
            mine[j] = i == l ? sum : mine[j];
        }
    });
    if (NG > 1) {
#pragma unroll
        for (int j = 0; j < V; j++) parts[(j * WAVES + wave) * 64 + lane] = mine[j];
        lh_lds_barrier();
        if (grp != 0) return;
#pragma unroll
        for (int j = 0; j < V; j++)
#pragma unroll
            for (int g = 1; g < NG; g++) mine[j] += parts[(j * WAVES + wave + g) * 64 + lane];
    }
    if constexpr (M == kGated) {
        const uint16_t mine16 = lh_f2h(mine[0]);
        uint32_t gate, up;
        lh_pair32_u(mine16, gate, up);
        if (lane < count) a.y[0][first + lane * step] = lh_gelu_mul_h((uint16_t)gate, (uint16_t)up);
    } else if (l < count) {
        const uint32_t q = first + l * step, pr = problem(q), row = 2 * (q - pr * pairs) + half;
        if (row < rows)
#pragma unroll
            for (int j = 0; j < V; j++)
                if (v0 + j < a.batch) reinterpret_cast<uint16_t*>(reinterpret_cast<char*>(a.y[pr]) + (size_t)(v0 + j) * a.ystride)[row] = M == kFactor ? lh_gelu_mul_h(lh_f2h(mine[j]), factor) : lh_f2h(mine[j]);
    }
}

}  // namespace

int lh_launch_matvec_direct(lh_context* ctx, lh_quant fmt, uint32_t count, const void* const* matrices, const void* vector, void* const* outputs, uint32_t rows,
                                uint32_t K, const XPrologue& pro, uint32_t batch, uint32_t xstride, uint32_t ystride, bool gated, const uint16_t* factor) {
    const uint32_t ng = (K + 2047) / 2048;
    if (count > 8 || ng > 6 || (batch > 1 && (count > 1 || pro.kind != kXProNone))) return -1;
    const uint32_t waves = (uint32_t)direct_waves((int)ng), teams = waves / ng;
    // Beyond 8 pairs of rows per wave of a workgroup per CU (16 where a row takes several waves) the unpacking is what takes the time, and
    // the matrix cores do the rest of the work for nothing: 65536 x 1536 (16 per wave) 13.1 us against 11.2 there, 32768 x 2048 (8) 8.3
    // against 8.7; 16384 x 12288 (16) 19.1 against 22.2.  The line does not depend on the batch: what a vector gives alone it gives in one.
    const uint64_t total = gated ? rows : (uint64_t)((rows + 1) / 2) * count, slots = (uint64_t)ctx->cu_count * teams;
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
    const uint32_t step = grid.x * teams;
    DirectArgs a{{}, {}, count, (rows + 1) / 2, (uint32_t)total, (uint32_t)(total / step), (uint32_t)(total % step), batch, xstride, ystride, pro.store, pro.eps, pro.scale, pro.tail,
                 pro.head_dim, pro.res != nullptr, pro.aux2 != nullptr, factor};
    for (uint32_t i = 0; i < count; i++) { a.m[i] = (const uint8_t*)matrices[i]; a.y[i] = (uint16_t*)outputs[i]; }
    const uint16_t* const self = (const uint16_t*)vector;
    const uint16_t* const second = pro.kind == kXProRotate ? (const uint16_t*)pro.signs : pro.aux;
    const size_t lds = (size_t)v * ng * 4096 + ((size_t)v * waves * 64 + 32) * 4;
    int r = LH_OK;
#define LH_DIRECT_V(FMT, KIND, NG, V, M)                                                                                                                     \
    do {                                                                                                                                                 \
        if (lds > 65536) r = lh_raise_dynamic_lds(ctx, (const void*)matvec_direct_kernel<FMT, KIND, NG, V, M>, lds, "matvec_quant");                         \
        if (r == LH_OK)                                                                                                                                  \
            hipLaunchKernelGGL((matvec_direct_kernel<FMT, KIND, NG, V, M>), grid, dim3(64 * waves), lds, ctx->stream, vector, second, pro.res ? pro.res : self, \
                               pro.aux2 ? pro.aux2 : self, a.m[0], K, rows, step, a);                                                                    \
    } while (0)
#define LH_DIRECT(FMT, KIND, NG)                                                            \
    do {                                                                                    \
        if constexpr (KIND == kXProNone) {                                                  \
            if constexpr (direct_waves(NG) <= 8) {                                          \
                if (v == 4) { LH_DIRECT_V(FMT, KIND, NG, 4, kOne); break; }                 \
            }                                                                               \
            if (v == 2) { LH_DIRECT_V(FMT, KIND, NG, 2, kOne); break; }                     \
        }                                                                                   \
        if constexpr (KIND == kXProRmsNorm) {                                               \
            if (gated) { LH_DIRECT_V(FMT, KIND, NG, 1, kGated); break; }                    \
            if (factor) { LH_DIRECT_V(FMT, KIND, NG, 1, kFactor); break; }                  \
        }                                                                                   \
        if (count > 1) LH_DIRECT_V(FMT, KIND, NG, 1, kSeveral);                             \
        else LH_DIRECT_V(FMT, KIND, NG, 1, kOne);                                           \
    } while (0)
#define LH_DIRECT_KIND(FMT, KIND)                  \
    do {                                           \
        switch (ng) {                              \
            case 1: LH_DIRECT(FMT, KIND, 1); break; \
            case 2: LH_DIRECT(FMT, KIND, 2); break; \
            case 3: LH_DIRECT(FMT, KIND, 3); break; \
            case 4: LH_DIRECT(FMT, KIND, 4); break; \
            case 5: LH_DIRECT(FMT, KIND, 5); break; \
            default: LH_DIRECT(FMT, KIND, 6); break; \
        }                                          \
    } while (0)
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
#undef LH_DIRECT_V
    return r != LH_OK ? r : lh_check_launch(fmt == LH_TQ2_0 ? "matvec_tq2_0" : "matvec_q4_0");
}
