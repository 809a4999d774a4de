// Attention over a short span of packed 2-bit TurboQuant codes: a sliding window's one token, or one token of each of some dozens of
// sequences, or the rows of a prompt's chunk.
//
// Same contract and the same arithmetic as attention_tq_mfma.hip (stands in for shaders/attention_flash_tq.metal:154-690): the level table as bit
// planes, queries and softmax weights in 16-bit fixed point as two int8 limbs, v_mfma_i32_16x16x64_i8.  What differs is who does what.  There a K wave
// and a V wave walk a chunk of positions with a hand-over after each 64, which is what long spans want; over 512 positions the walk of three hand-overs is
// a chain of 7 of the launch's 10.7 us, on one CU.  Here:
//   * a wave takes an aligned group of 64 positions through both products, so that a window of 512 (nine groups) is one step of nine waves, and
//     nothing is handed over: a wave's softmax reference, sums and fixed-point scales are its own and meet in LDS at the end;
//   * a query's workgroups, four of them on four CUs, take 64 of the 256 output dims each (two with 128 where there are queries for that, or one with all).
//     Each repeats the scores (half of the work), none waits for another, and the kernel's output is final: no partial records, no merge launch;
//   * everything that comes from memory -- queries, codes of both kinds, norms -- is requested at the top, ahead of the level table, on which the
//     rest depends.
// Bound by the chain of one group and by a SIMD's two or three waves taking turns to issue.  From the first to the last instruction of one token over a
// window of 512: 10.7 us there, 6.1 here.  Recorded launches one after the other, a window of 512: 1 query 10.1 us there and 7.2, 64 lanes 11.9 and 8.1, 256 rows 11.2 and 9.8.
#include "attention_tq.hpp"
#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace {
using namespace lh_attn;

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef unsigned short us2_t __attribute__((ext_vector_type(2)));
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

constexpr uint32_t kGroup = 64, kHeads = 8, kDim = 256, kMaxWaves = 12;
constexpr float kLog2e = 1.4426950408889634f, kQmax = 32639.0f, kNoRef = -1.0e30f;

__device__ __forceinline__ u32x4_t ld16(const uint8_t* p) {
    typedef u32x4_t __attribute__((aligned(4))) u32x4_a4;
    return *reinterpret_cast<const u32x4_a4*>(p);
}

struct ShortShared {
    float queries[4][kHeads * 72 + 16];  // by field, head and code byte (a row in 72: a quarter wave's 16-byte reads on distinct banks; 16 more: the fields of a byte too)
    __device__ __forceinline__ float& q(uint32_t field, uint32_t head, uint32_t byte) { return queries[field][head * 72 + byte]; }
    uint8_t rqop[12][64][16];            // score operands per (plane, field) and lane
    float maxabs[kHeads], sum[kHeads];
    float fin_r[kMaxWaves][kHeads], fin_l[kMaxWaves][kHeads];
    float none[kDim];                    // zeros
};
// S: workgroups of a query, 256 / S output dims each.
template <int S>
struct ShortWave {
    float2 norm[kGroup];                 // (norm_k log2 e, norm_v) per position
    union {
        struct { uint8_t wx[3][1024], vt[4 / S][kGroup * 16]; };
        float park[kHeads][kDim / S];    // the wave's sums, when it is done
    };
};

// What a wave has requested of a group: see the loads in the kernel.
template <int S>
struct Group { u32x4_t k[4], v[4 / S]; uint32_t nk, nv; uint32_t lo, hi; };

// Walsh-Hadamard transform of a head of 64 N dims in a wave, a lane with dims lane + 64 j, pairs as in lh_fwht_lds.
template <int N>
__device__ __forceinline__ void transform_head(float (&v)[N], uint32_t lane) {
#pragma unroll
    for (int j = 0; j < N; j++) {
        v[j] = lh_fwht_lane_stage<1>(v[j], lane);
        v[j] = lh_fwht_lane_stage<2>(v[j], lane);
        v[j] = lh_fwht_lane_stage<4>(v[j], lane);
        v[j] = lh_fwht_lane_stage<8>(v[j], lane);
        v[j] = lh_fwht_lane_stage<16>(v[j], lane);
        v[j] = lh_fwht_lane_stage<32>(v[j], lane);
    }
#pragma unroll
    for (int s = 1; s < N; s *= 2)
#pragma unroll
        for (int j = 0; j < N; j++) {
            if (j & s) continue;
            const float a = v[j], b = v[j | s];
            v[j] = __fadd_rn(a, b);
            v[j | s] = __fsub_rn(a, b);
        }
}

// Where finished heads go as f16 behind the rotation out of code space, as hadamard_rotate_kernel makes it (a workgroup with all dims of a query).
struct RotateOut { uint16_t* out; const float (&sign)[4]; float inv_sqrt_d; };
struct NoRotation {};

template <int NPL, int S, class Load, class Rotation>
__device__ __forceinline__ void short_body(const AttnPointers& a, const AttnParams& p, ShortShared& sh, ShortWave<S>& mine, Group<S> gr, uint32_t G, uint32_t g_last, Load load,
                                           float alpha, float beta, float gam, float delta, uint32_t qi, uint32_t kvh, uint32_t group, uint32_t nwaves, uint32_t parts, const Rotation& rotation) {
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), pcol = lane & 15, g = lane >> 4;
    constexpr int E = 4 / S;              // chunks of 16 code bytes, 64 dims
    if (wave == nwaves - 1)
#pragma unroll
        for (int e = 0; e < E; e++) sh.none[64 * e + lane] = 0.0f;
    const float cmax = fmaxf(fmaxf(fabsf(beta), fabsf(0.5f * gam)), NPL == 3 ? fabsf(delta) : 0.0f), inv_cmax = cmax > 0.0f ? 1.0f / cmax : 0.0f;

    // ---- score operands: row r of the product is head (r / 4) + 4 ((r / 2) % 2), limb r % 2; k slot (word m, byte e) of row group g is code byte
    //      16 g + 4 m + e, i.e. dim 4 (16 g + 4 m + e) + f for field f.  The lanes of a head's two limbs quantise two of the four words each.
    {
        const uint32_t h = (pcol >> 2) + 4 * ((pcol >> 1) & 1), limb = pcol & 1;
        const float ma = sh.maxabs[h], inv = (ma > 0.0f && cmax > 0.0f) ? kQmax / (ma * cmax) : 0.0f;
        for (uint32_t unit = wave; unit < 4 * NPL; unit += nwaves) {
            const uint32_t pl = unit >> 2, f = unit & 3;
            const float mul = (pl == 0 ? beta : pl == 1 ? 0.5f * gam : delta) * inv;
            uint32_t w[4];
#pragma unroll
            for (int mm = 0; mm < 2; mm++) {                  // word 2 mm + limb
                const float4 x = *reinterpret_cast<const float4*>(&sh.q(f, h, 16 * g + 4 * (2 * mm + limb)));
                const float xs[4] = {x.x, x.y, x.z, x.w};
                uint32_t lo = 0u, hi = 0u;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int n = (int)fminf(fmaxf(__builtin_rintf(xs[e] * mul), -kQmax), kQmax), low = (int)(int8_t)(n & 0xFF);
                    lo |= (uint32_t)(low & 0xFF) << (8 * e);
                    hi |= (uint32_t)(((n - low) >> 8) & 0xFF) << (8 * e);
                }
                const uint32_t own = limb ? hi : lo, got = (uint32_t)lh_dpp_i<LH_DPP_QUAD_XOR1>((int)(limb ? lo : hi));
                w[2 * mm] = limb ? got : own;
                w[2 * mm + 1] = limb ? own : got;
            }
            *reinterpret_cast<u32x4_t*>(&sh.rqop[unit][lane][0]) = (u32x4_t){w[0], w[1], w[2], w[3]};
        }
    }
    lh_lds_barrier();

    float R[2] = {kNoRef, kNoRef}, l_run[2] = {0.f, 0.f}, w_run[2] = {0.f, 0.f}, sctr[2] = {0.f, 0.f}, out[E][4][2];
#pragma unroll
    for (int e = 0; e < E; e++)
#pragma unroll
        for (int f = 0; f < 4; f++) out[e][f][0] = out[e][f][1] = 0.0f;
    const bool any = G <= g_last;
    if (any) {
        float cs[2], ca[2];              // logit (log2 domain) = norm_k log2 e (cs int + ca) for the lane's two heads g, g + 4
#pragma unroll
        for (int hs = 0; hs < 2; hs++) { cs[hs] = sh.maxabs[g + 4 * hs] * cmax * (0.25f / kQmax); ca[hs] = alpha * sh.sum[g + 4 * hs]; }
        v4i kept[4];                     // plane 0's, where there is room for them
#pragma unroll
        for (int u = 0; u < 4; u++) if (E == 1) kept[u] = *reinterpret_cast<const v4i*>(&sh.rqop[u][lane][0]);
        uint32_t from = lane;
        auto rq = [&](int u) { return E == 1 && u < 4 ? kept[u & 3] : *reinterpret_cast<const v4i*>(&sh.rqop[u][from][0]); };
        for (;;) {
            asm volatile("" : "+v"(from));                       // (or the operands would be read ahead of the loop and spilled)
            const bool valid = lane >= gr.lo && lane < gr.hi;
            mine.norm[lane] = make_float2(lh_h2f((uint16_t)gr.nk) * kLog2e, valid ? lh_h2f((uint16_t)gr.nv) : 0.0f);
#pragma unroll
            for (int e = 0; e < E; e++) *reinterpret_cast<u32x4_t*>(&mine.vt[e][lane * 16]) = gr.v[e];
            __builtin_amdgcn_wave_barrier();
            // ---- scores of 4 tiles x (this lane's column position, heads g and g + 4)
            float lg[4][2], vn[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                v4i acc1 = (v4i){0, 0, 0, 0}, acc4 = (v4i){0, 0, 0, 0};      // by mask scale: fields 0, 2 arrive x1, fields 1, 3 x4
                const uint32_t w[4] = {gr.k[q].x, gr.k[q].y, gr.k[q].z, gr.k[q].w};
#pragma unroll
                for (int pl = 0; pl < NPL; pl++) {
                    // plane 0 at bit 2 f of a field, plane 1 at bit 2 f + 1 (its coefficient is halved), plane 2 = bit0 & bit1 at bit 2 f
                    const uint32_t bits = pl == 1 ? 0x02020202u : 0x01010101u;
                    v4i b[4];
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        const uint32_t t = pl == 2 ? w[m] & (w[m] >> 1) : w[m], u = t >> 4;
                        b[0][m] = (int)(t & bits); b[1][m] = (int)(t & bits << 2); b[2][m] = (int)(u & bits); b[3][m] = (int)(u & bits << 2);
                    }
                    acc1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(rq(4 * pl), b[0], acc1, 0, 0, 0);
                    acc4 = __builtin_amdgcn_mfma_i32_16x16x64_i8(rq(4 * pl + 1), b[1], acc4, 0, 0, 0);
                    acc1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(rq(4 * pl + 2), b[2], acc1, 0, 0, 0);
                    acc4 = __builtin_amdgcn_mfma_i32_16x16x64_i8(rq(4 * pl + 3), b[3], acc4, 0, 0, 0);
                }
                const float2 nrm = mine.norm[16 * q + pcol];
                vn[q] = nrm.y;
                const bool in = 16 * q + pcol >= gr.lo && 16 * q + pcol < gr.hi;
#pragma unroll
                for (int hs = 0; hs < 2; hs++) {
                    const uint32_t t1 = ((uint32_t)acc1[2 * hs + 1] << 8) + (uint32_t)acc1[2 * hs], t4 = ((uint32_t)acc4[2 * hs + 1] << 8) + (uint32_t)acc4[2 * hs];
                    lg[q][hs] = in ? nrm.x * ((float)(int)((t1 << 2) + t4) * cs[hs] + ca[hs]) : -INFINITY;
                }
                __builtin_amdgcn_sched_barrier(0);           // (four tiles' operands at a time would not fit the registers)
            }
            // (all dims of a query at once leave no registers for another group: launched only where a wave has one)
            const bool more = S > 1 && G + nwaves <= g_last;
            if (E == 1 && more) gr = load(G + nwaves);       // (with more dims only when the registers are free)
            // ---- softmax weights relative to the wave's largest score so far, and as 16-bit fixed point relative to the head's largest weight of the group
            float wm[2] = {0.f, 0.f}, un[2], ww[4][2];
#pragma unroll
            for (int hs = 0; hs < 2; hs++) {
                const float r = fmaxf(R[hs], lh_group_max(fmaxf(fmaxf(lg[0][hs], lg[1][hs]), fmaxf(lg[2][hs], lg[3][hs])), 16)), fsc = __builtin_amdgcn_exp2f(R[hs] - r);
                l_run[hs] *= fsc; w_run[hs] *= fsc; sctr[hs] *= fsc;
#pragma unroll
                for (int e = 0; e < E; e++)
#pragma unroll
                    for (int f = 0; f < 4; f++) out[e][f][hs] *= fsc;
                R[hs] = r;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float ew = __builtin_amdgcn_exp2f(lg[q][hs] - r);
                    ww[q][hs] = ew * vn[q];
                    l_run[hs] += ew;
                    if constexpr (NPL == 3) w_run[hs] += ww[q][hs];
                    wm[hs] = fmaxf(wm[hs], fabsf(ww[q][hs]));
                }
                // The largest weight becomes the largest number (in the other kernel a power of two takes it into [0.5, 1): here a group is never cut by a
                // chunk's end into smaller ones with scales of their own, and the bit makes up for that.  Against 64 bits, a window of 300: 8.0e-5 there, 6.0e-5
                // here; of 512: 8.8e-5 and 6.1e-5).  Zero, subnormal or non-finite maximum: scale and step 0, as there.
                const uint32_t top = lh_group_max_u(__float_as_uint(wm[hs]), 16), e = top & 0x7F800000u;
                const bool ok = e != 0u && e < (253u << 23);
                const float sc = ok ? __builtin_amdgcn_rcpf(__uint_as_float(top)) : 0.0f;
                un[hs] = ok ? __uint_as_float(top) * (cmax * (1.0f / kQmax)) : 0.0f;
                const uint32_t A_ = pcol >> 2, B_ = ((pcol & 3) + 2 * (pcol >> 2)) & 3;      // k group and word: where the V codes of positions 16 q + pcol land
#pragma unroll
                for (int pl = 0; pl < NPL; pl++) {
                    const float c = (pl == 0 ? beta : pl == 1 ? 0.5f * gam : delta) * inv_cmax * (kQmax / 32767.0f) * sc;
                    const uint32_t p01 = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pknorm_i16(ww[0][hs] * c, ww[1][hs] * c));
                    const uint32_t p23 = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pknorm_i16(ww[2][hs] * c, ww[3][hs] * c));
                    const uint32_t t01 = __builtin_bit_cast(uint32_t, (us2_t)(__builtin_bit_cast(us2_t, p01) + (us2_t){0x80, 0x80})) ^ 0x00800080u;
                    const uint32_t t23 = __builtin_bit_cast(uint32_t, (us2_t)(__builtin_bit_cast(us2_t, p23) + (us2_t){0x80, 0x80})) ^ 0x00800080u;
                    uint8_t* dst = &mine.wx[pl][(16 * A_ + 4 * g + 2 * hs) * 16 + 4 * B_];
                    *reinterpret_cast<uint32_t*>(dst) = __builtin_amdgcn_perm(t23, t01, 0x06040200u);        // low limbs of tiles 0..3
                    *reinterpret_cast<uint32_t*>(dst + 16) = __builtin_amdgcn_perm(t23, t01, 0x07050301u);   // high limbs
                }
            }
            __builtin_amdgcn_wave_barrier();
            // ---- the values: one code byte over the positions of an operand word by transposing reads
            typedef __attribute__((address_space(3))) uint8_t* lds8_t;
            typedef __attribute__((address_space(3))) v2i* lds_v2i_t;
            v4i wop[NPL], csum = (v4i){0, 0, 0, 0};
#pragma unroll
            for (int pl = 0; pl < NPL; pl++) {
                wop[pl] = *reinterpret_cast<const v4i*>(&mine.wx[pl][lane * 16]);
                const int cb = pl == 0 ? 0x02020202 : pl == 1 ? 0x04040404 : 0x01010101;
                csum = __builtin_amdgcn_mfma_i32_16x16x64_i8(wop[pl], (v4i){cb, cb, cb, cb}, csum, 0, 0, 0);
            }
            const uint32_t i = lane & 15, A_ = lane >> 4, j = i >> 1;
#pragma unroll
            for (int e = 0; e < E; e++) {
                const lds8_t vt = (lds8_t)&mine.vt[e][0];
                uint32_t y[4];
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const uint32_t B_ = 2 * t + (j >> 2), src = 16 * (j & 3) + 4 * A_ + ((B_ + 2 * A_) & 3);
                    const v2i r = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i_t)(vt + src * 16 + 8 * (i & 1)));
                    y[2 * t] = (uint32_t)r.x;
                    y[2 * t + 1] = (uint32_t)r.y;
                }
                v4i acc[4];
#pragma unroll
                for (int f = 0; f < 4; f++) acc[f] = (v4i){0, 0, 0, 0};
#pragma unroll
                for (int pl = 0; pl < NPL; pl++)
#pragma unroll
                    for (int f = 0; f < 4; f++) {                            // field 3 is taken at field 2's place: 0x80 would be a negative int8
                        const uint32_t mask = (pl == 1 ? 0x02020202u : 0x01010101u) << (f == 3 ? 4 : 2 * f);
                        v4i b;
#pragma unroll
                        for (int m = 0; m < 4; m++) {
                            const uint32_t yp = pl == 2 ? y[m] & (y[m] >> 1) : y[m];
                            b[m] = (int)((f == 3 ? yp >> 2 : yp) & mask);
                        }
                        acc[f] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wop[pl], b, acc[f], 0, 0, 0);
                    }
#pragma unroll
                for (int hs = 0; hs < 2; hs++)
#pragma unroll
                    for (int f = 0; f < 4; f++) {
                        const int t = (int)(((uint32_t)acc[f][2 * hs + 1] << 8) + (uint32_t)acc[f][2 * hs]);
                        out[e][f][hs] = __builtin_fmaf((float)t, un[hs] * (f == 0 ? 1.0f : f == 1 ? 0.25f : 0.0625f), out[e][f][hs]);
                    }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int hs = 0; hs < 2; hs++) {
                const int t = (int)(((uint32_t)csum[2 * hs + 1] << 8) + (uint32_t)csum[2 * hs]);
                sctr[hs] = __builtin_fmaf((float)t, 0.25f * un[hs], sctr[hs]);
            }
            if (!more) break;
            G += nwaves;
            if (E > 1) gr = load(G);
            __builtin_amdgcn_wave_barrier();
        }
    }
    // ---- the wave's sums (in place of its operands, which it has read), then all waves'
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int hs = 0; hs < 2; hs++) {
        const uint32_t h = g + 4 * hs;
        const float l = lh_group_sum(l_run[hs], 16), w = NPL == 3 ? lh_group_sum(w_run[hs], 16) : 0.0f;
        if (pcol == 0) { sh.fin_l[wave][h] = l; sh.fin_r[wave][h] = R[hs] <= 0.5f * kNoRef ? -INFINITY : R[hs]; }
        const float bias = NPL == 3 ? (alpha + 0.5f * (beta + gam) + 0.25f * delta) * w - sctr[hs] : -sctr[hs];
#pragma unroll
        for (int e = 0; e < E; e++)
            *reinterpret_cast<float4*>(&mine.park[h][64 * e + 4 * pcol]) = make_float4(out[e][0][hs] + bias, out[e][1][hs] + bias, out[e][2][hs] + bias, out[e][3][hs] + bias);
    }
    lh_lds_barrier();
    if (wave >= group) return;
    const float r = lane < parts ? sh.fin_r[lane][wave] : -INFINITY, top = lh_group_max(r, 16);
    const float f = r == -INFINITY ? 0.0f : exp2f(r - top), l = lh_group_sum(lane < parts ? f * sh.fin_l[lane][wave] : 0.0f, 16);
    const ShortWave<S>* const all = &mine - wave;
    float o[E] = {};
    for (uint32_t w0 = 0; w0 < parts; w0 += 4) {                // (one at a time each is a trip to LDS; past the last: zeros)
        float x[4][E];
#pragma unroll
        for (uint32_t u = 0; u < 4; u++) {
            const float* const sums = w0 + u < parts ? all[w0 + u].park[wave] : sh.none;
#pragma unroll
            for (int e = 0; e < E; e++) x[u][e] = sums[64 * e + lane];
        }
#pragma unroll
        for (uint32_t u = 0; u < 4; u++) {
            const float fw = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(f), (int)(w0 + u)));
#pragma unroll
            for (int e = 0; e < E; e++) o[e] = __builtin_fmaf(fw, x[u][e], o[e]);
        }
    }
    const float total = __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(l)));
    const size_t at = ((size_t)qi * p.num_q_heads + kvh * group + wave) * kDim + kDim / S * blockIdx.x + lane;
#pragma unroll
    for (int e = 0; e < E; e++) o[e] = total > 0.0f ? o[e] / total : 0.0f;
    if constexpr (std::is_same_v<Rotation, RotateOut>) {
        static_assert(E == 4, "all dims of a head");
        transform_head(o, lane);
#pragma unroll
        for (int e = 0; e < E; e++) rotation.out[at + 64 * e] = lh_f2h_exact(__fmul_rn(__fmul_rn(o[e], rotation.inv_sqrt_d), rotation.sign[e]));
    } else {
#pragma unroll
        for (int e = 0; e < E; e++) a.out[at + 64 * e] = o[e];
    }
}

// The codes and norms of group G_ of positions [lo, hi).  Lanes whose position is not visible read one that is: nothing of it is used (its weight is zero).
template <int S>
__device__ __forceinline__ Group<S> load_group(const AttnPointers& a, const AttnParams& p, uint32_t G_, uint32_t lo, uint32_t hi, uint32_t lane_base, uint32_t kv_heads, uint32_t kvh) {
    Group<S> r;
    const uint32_t stride = kv_heads * 64;
    uint32_t at_lane = threadIdx.x & 63;
    asm volatile("" : "+v"(at_lane));                           // (a second group's addresses are not to wait in registers for the rare loop that needs them)
    const uint32_t start = G_ << 6, base = lane_base + (p.ring_capacity ? start % p.ring_capacity : start);
    r.lo = lo > start ? lo - start : 0u;
    r.hi = std::min(hi - start, kGroup);
    auto at = [&](uint32_t i) { return (size_t)(base + std::min(std::max(i, r.lo), r.hi - 1)); };
#pragma unroll
    for (int q = 0; q < 4; q++) r.k[q] = ld16(a.k_codes + at(16 * q + (at_lane & 15)) * stride + kvh * 64 + 16 * (at_lane >> 4));
    r.nk = a.k_norms[at(at_lane) * kv_heads + kvh];
    r.nv = a.v_norms[at(at_lane) * kv_heads + kvh];
#pragma unroll
    for (int e = 0; e < 4 / S; e++) r.v[e] = ld16(a.v_codes + at(at_lane) * stride + kvh * 64 + 16 * (4 / S * blockIdx.x + e));
    return r;
}

// L[c] = alpha + beta bit0 + gam bit1 + delta bit0 bit1: as in attention_tq_mfma_kernel
template <int S, class Load, class Rotation>
__device__ __forceinline__ void short_by_levels(const AttnPointers& a, const AttnParams& p, ShortShared& sh, ShortWave<S>& mine, const Group<S>& first, uint32_t begin, uint32_t end, Load load,
                                                float L0, float L1, float L2, float L3, uint32_t qi, uint32_t kvh, uint32_t group, uint32_t nwaves, uint32_t parts, const Rotation& rotation) {
    const float d_raw = (L3 - L2) - (L1 - L0), lmax = fmaxf(fmaxf(fabsf(L0), fabsf(L1)), fmaxf(fabsf(L2), fabsf(L3))), l_mean = 0.25f * ((L0 + L3) + (L1 + L2));
    if (fabsf(d_raw) > 1e-5f * lmax || fabsf(l_mean) > 1e-6f * lmax) short_body<3, S>(a, p, sh, mine, first, begin, end, load, L0, L1 - L0, L2 - L0, d_raw, qi, kvh, group, nwaves, parts, rotation);
    else short_body<2, S>(a, p, sh, mine, first, begin, end, load, L0 - 0.25f * d_raw, (L1 - L0) + 0.5f * d_raw, (L2 - L0) + 0.5f * d_raw, 0.0f, qi, kvh, group, nwaves, parts, rotation);
}

__device__ __forceinline__ float level_of(float table, int i) { return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(table), i)); }

// The raw values of a head: the splits in order, in f32, rounded to f16 as decode_qkv_prepare_kernel does, or finished rows (a lane's first value at `raw`).
template <int N>
__device__ __forceinline__ void raw_head(uint16_t (&h)[N], const TokenPrep& t, uint32_t row, uint32_t column, const uint16_t* raw, uint32_t lane) {
    if (t.partial) {
        const size_t zstride = (size_t)t.rows * t.part_cols;
        const float* part = t.partial + (size_t)row * t.part_cols + column + lane;
        float acc[N] = {};
        for (uint32_t z0 = 0; z0 < t.splits; z0 += 8) {
            float x[8][N];
#pragma unroll
            for (uint32_t u = 0; u < 8; u++)
#pragma unroll
                for (int j = 0; j < N; j++) x[u][j] = part[(size_t)(z0 + u < t.splits ? z0 + u : t.splits - 1) * zstride + 64 * j];
#pragma unroll
            for (uint32_t u = 0; u < 8; u++)
#pragma unroll
                for (int j = 0; j < N; j++) if (z0 + u < t.splits) acc[j] += x[u][j];
        }
#pragma unroll
        for (int j = 0; j < N; j++) h[j] = lh_f2h(acc[j]);
    } else {
#pragma unroll
        for (int j = 0; j < N; j++) h[j] = raw[64 * j];
    }
}
// The codes of a head, four to a byte.
template <int N>
__device__ __forceinline__ void store_codes(uint8_t* bytes, const uint32_t (&code)[N], uint32_t lane) {
#pragma unroll
    for (int j = 0; j < N; j++) {
        uint32_t b = code[j] << 2 * (lane & 3);
        b |= (uint32_t)lh_dpp_i<LH_DPP_QUAD_XOR1>((int)b);
        b |= (uint32_t)lh_dpp_i<LH_DPP_QUAD_XOR2>((int)b);
        if ((lane & 3) == 0) bytes[(lane >> 2) + 16 * j] = (uint8_t)b;
    }
}

// The leading arguments arrive in registers with the wave (see the Makefile); the structures repeat them.
template <int S>
__global__ __launch_bounds__(64 * kMaxWaves) void attention_tq_short_kernel(const float* queries, const float* levels, uint32_t q_heads, uint32_t kv_heads, const AttnPointers a,
                                                                            const AttnParams p) {
    extern __shared__ __align__(16) uint8_t lds[];
    ShortShared& sh = *reinterpret_cast<ShortShared*>(lds);
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nwaves = blockDim.x >> 6;
    ShortWave<S>& mine = reinterpret_cast<ShortWave<S>*>(lds + sizeof(ShortShared))[wave];
    uint32_t qi = blockIdx.y, kvh = 0, group = q_heads;
    if (kv_heads != 1) { qi = blockIdx.y / kv_heads; kvh = blockIdx.y - qi * kv_heads; group = q_heads / kv_heads; }
    // ---- a wave has a head of the query
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (wave < group) x = reinterpret_cast<const float4*>(queries + ((size_t)qi * q_heads + kvh * group + wave) * kDim)[lane];
    const float table = levels[lane & 3];                       // (as a scalar load every argument behind it would wait for it)

    uint32_t lo, hi, lane_base;
    query_range(p, a.positions, qi, lo, hi, lane_base);
    const uint32_t G = (lo >> 6) + wave, g_last = hi > lo ? (hi - 1) >> 6 : 0u;
    const bool none = hi <= lo;
    auto load = [&](uint32_t G_) { return load_group<S>(a, p, G_, lo, hi, lane_base, kv_heads, kvh); };
    Group<S> first{};
    if (!none && G <= g_last) first = load(G);

    // ---- per head: max |q| (quantisation scale) and sum (constant term of the level table)
    if (wave < kHeads) {
        sh.q(0, wave, lane) = x.x; sh.q(1, wave, lane) = x.y; sh.q(2, wave, lane) = x.z; sh.q(3, wave, lane) = x.w;
        const float m = lh_group_max(fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w))), 64), s = lh_group_sum((x.x + x.y) + (x.z + x.w), 64);
        if (lane == 0) { sh.maxabs[wave] = m; sh.sum[wave] = s; }
    }
    lh_lds_barrier();
    short_by_levels<S>(a, p, sh, mine, first, none ? 1u : G, none ? 0u : g_last, load, level_of(table, 0), level_of(table, 1), level_of(table, 2), level_of(table, 3), qi, kvh, group,
                       nwaves, nwaves, NoRotation{});
}

// ---- the query's own preparation in the same launch -------------------------------------------------------------------------------
// A token's preparation (6.7 us; 5.0 without a key and a value) and its attention over a window (7.3) are two chains on a few CUs, one behind
// the other, and each begins with a trip to memory.  In one launch 9.5 us (9.2), a token at 32768 positions with eight such layers 577 -> 547.  Here a workgroup prepares its query itself: the head that a wave stages it also norms,
// turns and transforms, in registers (a lane has dims lane + 64 j: a rotary pair is one lane's, and so are the transform's last two
// stages).  The position's own key and value need a chain of 256 dependent additions for their codes: two more waves walk it while
// the others are at the groups before it, and leave their one position as a partial result of its own (its score, the value's levels,
// weight 1) that the last step merges with the rest; they walk it between the others' barriers, and store behind the last one (with all of it behind
// the score operands they were 1.6 us longer than the groups).  Every workgroup of a query repeats this; the first one also stores what the
// preparation leaves: f16 heads, codes, norms.  Same operations in the same order as decode_qkv_prepare_kernel: the same bits.
struct TokenShared {
    float2 turn[kDim / 2];               // cosine and sine of a rotary pair
    float square[2][kDim];
};

// One head in a wave: h[j] becomes the f16 value of dim lane + 64 j behind the norm.
template <int N>
__device__ __forceinline__ void norm_head(uint16_t (&h)[N], const uint16_t (&w)[N], bool weighted, float eps) {
    float total = 0.0f, s[N];
#pragma unroll
    for (int j = 0; j < N; j++) {
        const float x = lh_h2f(h[j]);
        float sq = x * x;
        asm volatile("" : "+v"(sq));                            // (rounded before it is added)
        s[j] = lh_group_sum(sq, 64);
    }
#pragma unroll
    for (int j = 0; j < N; j++) total += s[j];
    const float rms = rsqrtf(total / (float)(64 * N) + eps);
#pragma unroll
    for (int j = 0; j < N; j++) h[j] = lh_f2h_exact(lh_norm_product(lh_h2f(h[j]), rms, weighted ? lh_h2f(w[j]) : 1.0f));
}
template <int N>
__device__ __forceinline__ void turn_head(uint16_t (&h)[N], const float2* turn, uint32_t angles, uint32_t lane) {
#pragma unroll
    for (int j = 0; j < N / 2; j++) {
        if (lane + 64 * j >= angles) continue;
        const float2 t = turn[lane + 64 * j];
        lh_rope_apply(lh_h2f(h[j]), lh_h2f(h[j + N / 2]), t.x, t.y, h[j], h[j + N / 2]);
    }
}
// The codes of a head and its norm, as encode_vector makes them (turboquant_kv.hip): the squares, their sum from left to right as the CPU
// encoder has it, the rest.
template <int N>
__device__ __forceinline__ void place_squares(const uint16_t (&h)[N], float* square, uint32_t lane) {
#pragma unroll
    for (int j = 0; j < N; j++) square[lane + 64 * j] = lh_h2f(h[j]) * lh_h2f(h[j]);
    __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ float add_squares(float sum, const float* square, uint32_t first, uint32_t count = kDim / 2) {       // half of them
#pragma unroll 8
    for (uint32_t i = first; i < first + count; i += 4) {
        const float4 q = *reinterpret_cast<const float4*>(&square[i]);
        sum += q.x; sum += q.y; sum += q.z; sum += q.w;
    }
    return sum;
}
template <int N>
__device__ __forceinline__ uint16_t encode_head(const uint16_t (&h)[N], float sum, const float (&sign)[N], const float (&level)[4], float inv_sqrt_d, uint32_t lane, uint32_t (&code)[N]) {
    const float norm = __fsqrt_rn(sum), inv = __fdiv_rn(1.0f, norm);
    float v[N];
#pragma unroll
    for (int j = 0; j < N; j++) {
        v[j] = lh_h2f(h[j]);
        if (norm > 0.0f) v[j] = __fmul_rn(v[j], inv);
        v[j] = __fmul_rn(v[j], sign[j]);
        asm volatile("" : "+v"(v[j]));
    }
    transform_head(v, lane);
#pragma unroll
    for (int j = 0; j < N; j++) {
        float y = __fmul_rn(v[j], inv_sqrt_d), best = INFINITY;
        asm volatile("" : "+v"(y));                             // (rounded before the levels are taken off)
        code[j] = 0;
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
            const float d = fabsf(__fsub_rn(y, level[i]));
            if (d < best) { best = d; code[j] = i; }
        }
    }
    return lh_f2h_exact(norm);
}

// The leading arguments arrive in registers with the wave (see the Makefile); the structures repeat them.
template <int S, bool OWN, bool ROTATE>
__global__ __launch_bounds__(64 * kMaxWaves) void attention_tq_token_kernel(const float* levels, const float* signs, uint32_t q_heads, uint32_t kv_heads, const AttnPointers a,
                                                                            const AttnParams p, const TokenPrep t) {
    extern __shared__ __align__(16) uint8_t lds[];
    ShortShared& sh = *reinterpret_cast<ShortShared*>(lds);
    TokenShared& ts = *reinterpret_cast<TokenShared*>(lds + sizeof(ShortShared));
    ShortWave<S>* const all = reinterpret_cast<ShortWave<S>*>(lds + sizeof(ShortShared) + sizeof(TokenShared));
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nall = blockDim.x >> 6, nwaves = OWN ? nall - 2 : nall;
    uint32_t qi = blockIdx.y, kvh = 0, group = q_heads;
    if (kv_heads != 1) { qi = blockIdx.y / kv_heads; kvh = blockIdx.y - qi * kv_heads; group = q_heads / kv_heads; }
    const bool own = OWN && wave >= nwaves, is_v = own && wave > nwaves, is_q = wave < group, works = is_q || own;      // (the first eight waves are no `own`)
    const float table = levels[lane & 3];                       // (as a scalar load every argument behind it would wait for it)

    // ---- the rotary pairs by two waves, the value's and the last of the others (a window's ninth has no head), ahead of what they wait for
    const uint32_t position = p.mode == kBatched ? a.positions[qi] : p.pos0, angles = (uint32_t)((float)kDim * t.prf) / 2;
    const uint32_t second = OWN ? nwaves - 1 : nall - 2;
    if (wave == nall - 1 || wave == second) {
        const uint32_t i = lane + (wave == second ? 64 : 0);
        float c = 1.0f, s = 0.0f;
        if (i < angles) lh_rope_cos_sin(i, kDim, position, t.theta, c, s);
        ts.turn[i] = make_float2(c, s);
    }

    // ---- the wave's head: raw values, norm weights, signs
    const uint32_t head = is_q ? kvh * group + wave : kvh, column = (is_q ? head : is_v ? q_heads + kv_heads + kvh : q_heads + kvh) * kDim;
    const size_t row_at = ((size_t)qi * (is_q ? q_heads : kv_heads) + head) * kDim + lane;
    const uint16_t* const norm_w = is_q ? t.q_norm : own && !is_v ? t.k_norm : nullptr;
    uint16_t h[4] = {0, 0, 0, 0}, w[4] = {0, 0, 0, 0};
    float sign[4];
    if (works) {
        raw_head(h, t, qi, column, (is_q ? t.q : is_v ? t.v : t.k) + row_at, lane);
        if (norm_w)
#pragma unroll
            for (int j = 0; j < 4; j++) w[j] = norm_w[lane + 64 * j];
    }
#pragma unroll
    for (int j = 0; j < 4; j++) sign[j] = signs[lane + 64 * j];

    uint32_t lo, hi, lane_base;
    query_range(p, a.positions, qi, lo, hi, lane_base);
    if (OWN) hi = hi > lo ? hi - 1 : hi;                        // the position itself comes from its own two waves
    const uint32_t G = (lo >> 6) + wave, g_last = hi > lo ? (hi - 1) >> 6 : 0u;
    const bool none = hi <= lo;
    auto load = [&](uint32_t G_) { return load_group<S>(a, p, G_, lo, hi, lane_base, kv_heads, kvh); };
    Group<S> first{};
    if (!own && !none && G <= g_last) first = load(G);

    if (works && (is_v || norm_w)) norm_head(h, w, !is_v, t.eps);
    lh_lds_barrier();
    if (works && !is_v) turn_head(h, ts.turn, angles, lane);
    if (works && blockIdx.x == 0) {
        uint16_t* const to = (is_q ? t.q_out : is_v ? t.v_out : t.k_out) + row_at;
#pragma unroll
        for (int j = 0; j < 4; j++) to[64 * j] = h[j];
    }
    if (wave < kHeads) {
        float x[4];
#pragma unroll
        for (int j = 0; j < 4; j++) { x[j] = is_q ? __fmul_rn(lh_h2f(h[j]), sign[j]) : 0.0f; asm volatile("" : "+v"(x[j])); }
        transform_head(x, lane);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            x[j] = __fmul_rn(x[j], t.inv_sqrt_d);
            asm volatile("" : "+v"(x[j]));
            sh.q(lane & 3, wave, (lane >> 2) + 16 * j) = x[j];
        }
        const float m = lh_group_max(fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3]))), 64), s = lh_group_sum((x[0] + x[1]) + (x[2] + x[3]), 64);
        if (lane == 0) { sh.maxabs[wave] = m; sh.sum[wave] = s; }
    }
    // The position's own waves walk their sums while the others are between barriers.
    float* const square = ts.square[is_v ? 1 : 0];
    float squares = 0.0f;
    if (OWN && own) { place_squares(h, square, lane); squares = add_squares(0.0f, square, 0); }
    lh_lds_barrier();
    const float L0 = level_of(table, 0), L1 = level_of(table, 1), L2 = level_of(table, 2), L3 = level_of(table, 3);
    if (!own) {
        const uint32_t parts = OWN ? nwaves + 1 : nwaves;
        if constexpr (ROTATE) short_by_levels<S>(a, p, sh, all[wave], first, none ? 1u : G, none ? 0u : g_last, load, L0, L1, L2, L3, qi, kvh, group, nwaves, parts, RotateOut{t.rotated, sign, t.inv_sqrt_d});
        else short_by_levels<S>(a, p, sh, all[wave], first, none ? 1u : G, none ? 0u : g_last, load, L0, L1, L2, L3, qi, kvh, group, nwaves, parts, NoRotation{});
        return;
    }
    if constexpr (OWN) {
        squares = add_squares(squares, square, kDim / 2);
        lh_lds_barrier();                                       // short_body's, behind the score operands
        const float level[4] = {L0, L1, L2, L3};
        uint32_t code[4];
        const uint16_t norm = encode_head(h, squares, sign, level, t.inv_sqrt_d, lane, code);
        float x[4];
#pragma unroll
        for (int j = 0; j < 4; j++) x[j] = code[j] == 0 ? L0 : code[j] == 1 ? L1 : code[j] == 2 ? L2 : L3;
        if (is_v) {
            constexpr uint32_t E = 4 / S;
            const float n = lh_h2f(norm);
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (j / E == blockIdx.x)
#pragma unroll
                    for (uint32_t i = 0; i < kHeads; i++) all[nwaves].park[i][64 * (j % E) + lane] = x[j] * n;
            if (lane < kHeads) sh.fin_l[nwaves][lane] = 1.0f;
        } else {                                                // eight lanes a head, eight code bytes each: the levels in the queries' order by way of LDS
            const uint32_t i = lane >> 3, byte = 8 * (lane & 7);
#pragma unroll
            for (int j = 0; j < 4; j++) square[(lane & 3) * 64 + (lane >> 2) + 16 * j] = x[j];
            __builtin_amdgcn_wave_barrier();
            float d = 0.0f;
#pragma unroll
            for (int f = 0; f < 4; f++)
#pragma unroll
                for (int c = 0; c < 8; c += 4) {
                    const float4 q = *reinterpret_cast<const float4*>(&sh.q(f, i, byte + c)), l = *reinterpret_cast<const float4*>(&square[f * 64 + byte + c]);
                    d = __builtin_fmaf(q.x, l.x, d); d = __builtin_fmaf(q.y, l.y, d); d = __builtin_fmaf(q.z, l.z, d); d = __builtin_fmaf(q.w, l.w, d);
                }
            d = lh_group_sum(d, 8);
            if ((lane & 7) == 0) sh.fin_r[nwaves][i] = d * (lh_h2f(norm) * kLog2e);
        }
        lh_lds_barrier();                                       // short_body's, ahead of the merge
        if (blockIdx.x != 0) return;
        const size_t slot = ((size_t)lane_base + (p.ring_capacity ? position % p.ring_capacity : position)) * kv_heads + kvh;
        store_codes((is_v ? t.v_codes : t.k_codes) + slot * (kDim / 4), code, lane);
        if (lane == 0) (is_v ? t.v_norms : t.k_norms)[slot] = norm;
    }
}

// The preparation by itself: a wave a head, in registers as above, a workgroup some heads of a row, or all of them, with the rotary pairs once.  What bounds many rows is
// vector instructions: with a workgroup a head and the pairs' cosines and sines in each of them decode_qkv_prepare_kernel took 13.0 us for 256 rows of 10 heads of 256 dims and 18.3
// of 512; now 7.3 and 10.0.  Few rows are bound by what a CU reads of the partial tiles, so that a
// workgroup takes fewer heads there (64 rows of 512 dims, with keys and values and without: 9.2 us on average with all heads, 7.8).  The same bits.
struct RowsPrep { float* rq; const float* levels; const uint32_t* positions; uint32_t position, ring_capacity, lane_capacity, q_heads, kv_heads; };
constexpr uint32_t kRowHeads = 16;
template <int N>
__global__ __launch_bounds__(64 * kRowHeads) void prepare_rows_kernel(const RowsPrep r, const TokenPrep t) {
    constexpr uint32_t D = 64 * N;
    __shared__ float2 turn[D / 2];
    extern __shared__ __align__(16) float squares[];            // [waves][D]
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), row = blockIdx.x, b = blockIdx.y * (blockDim.x >> 6) + wave;
    const bool is_q = b < r.q_heads, is_v = b >= r.q_heads + r.kv_heads, works = b < r.q_heads + 2 * r.kv_heads;
    const uint32_t head = is_q ? b : is_v ? b - r.q_heads - r.kv_heads : b - r.q_heads;
    const size_t row_at = ((size_t)row * (is_q ? r.q_heads : r.kv_heads) + head) * D + lane;
    const uint16_t* const norm_w = is_q ? t.q_norm : is_v ? nullptr : t.k_norm;
    uint16_t h[N] = {}, w[N] = {};
    float sign[N];
    if (works) raw_head(h, t, row, b * D, (is_q ? t.q : is_v ? t.v : t.k) + row_at, lane);
    if (norm_w)
#pragma unroll
        for (int j = 0; j < N; j++) w[j] = norm_w[lane + 64 * j];
#pragma unroll
    for (int j = 0; j < N; j++) sign[j] = t.signs[lane + 64 * j];
    const float table = works && !is_q ? r.levels[lane & 3] : 0.0f;        // (null where there are queries alone)
    const uint32_t position = r.positions ? r.positions[row] : r.position + row, angles = (uint32_t)((float)D * t.prf) / 2;
    for (uint32_t i = tid; i < D / 2; i += blockDim.x) {
        float c = 1.0f, s = 0.0f;
        if (i < angles) lh_rope_cos_sin(i, D, position, t.theta, c, s);
        turn[i] = make_float2(c, s);
    }
    if (is_v || norm_w) norm_head(h, w, !is_v, t.eps);
    lh_lds_barrier();
    if (!works) return;
    if (!is_v) turn_head(h, turn, angles, lane);
    uint16_t* const to = (is_q ? t.q_out : is_v ? t.v_out : t.k_out) + row_at;
#pragma unroll
    for (int j = 0; j < N; j++) to[64 * j] = h[j];
    if (is_q) {
        float x[N];
#pragma unroll
        for (int j = 0; j < N; j++) { x[j] = __fmul_rn(lh_h2f(h[j]), sign[j]); asm volatile("" : "+v"(x[j])); }
        transform_head(x, lane);
#pragma unroll
        for (int j = 0; j < N; j++) r.rq[row_at + 64 * j] = __fmul_rn(x[j], t.inv_sqrt_d);
        return;
    }
    float* const square = squares + wave * D;
    place_squares(h, square, lane);
    const float sum = add_squares(0.0f, square, 0, D);
    const float level[4] = {level_of(table, 0), level_of(table, 1), level_of(table, 2), level_of(table, 3)};
    uint32_t code[N];
    const uint16_t norm = encode_head(h, sum, sign, level, t.inv_sqrt_d, lane, code);
    const size_t slot = ((size_t)row * r.lane_capacity + (r.ring_capacity ? position % r.ring_capacity : position)) * r.kv_heads + head;
    store_codes((is_v ? t.v_codes : t.k_codes) + slot * (D / 4), code, lane);
    if (lane == 0) (is_v ? t.v_norms : t.k_norms)[slot] = norm;
}

template <int S> constexpr size_t short_lds(uint32_t waves) { return sizeof(ShortShared) + waves * sizeof(ShortWave<S>); }

template <int S>
int launch(lh_context* ctx, const char* op, const AttnPointers& a, const AttnParams& p, uint32_t waves) {
    hipLaunchKernelGGL(attention_tq_short_kernel<S>, dim3(S, p.num_queries * p.num_kv_heads), dim3(64 * waves), short_lds<S>(waves), ctx->stream, a.rq, a.levels,
                       p.num_q_heads, p.num_kv_heads, a, p);
    return lh_check_launch(op);
}

template <int S> constexpr size_t token_lds(uint32_t waves) { return sizeof(TokenShared) + short_lds<S>(waves); }

template <int S, bool ROTATE = false>
int launch_token_form(lh_context* ctx, const char* op, const AttnPointers& a, const AttnParams& p, const TokenPrep& t, uint32_t waves) {
    const dim3 grid(S, p.num_queries * p.num_kv_heads);
    if (t.k_codes) hipLaunchKernelGGL((attention_tq_token_kernel<S, true, ROTATE>), grid, dim3(64 * (waves + 2)), token_lds<S>(waves + 2), ctx->stream, a.levels, t.signs, p.num_q_heads, p.num_kv_heads, a, p, t);
    else hipLaunchKernelGGL((attention_tq_token_kernel<S, false, ROTATE>), grid, dim3(64 * waves), token_lds<S>(waves), ctx->stream, a.levels, t.signs, p.num_q_heads, p.num_kv_heads, a, p, t);
    return lh_check_launch(op);
}

}  // namespace

int lh_attention_short_init(lh_context* ctx) {
    int r = lh_raise_dynamic_lds(ctx, (const void*)attention_tq_short_kernel<4>, short_lds<4>(kMaxWaves), "context_create");
    if (r == LH_OK) r = lh_raise_dynamic_lds(ctx, (const void*)attention_tq_short_kernel<2>, short_lds<2>(kMaxWaves), "context_create");
    if (r == LH_OK) r = lh_raise_dynamic_lds(ctx, (const void*)attention_tq_short_kernel<1>, short_lds<1>(kMaxWaves), "context_create");
    const auto raise = [&](auto kernel, size_t bytes) { if (r == LH_OK) r = lh_raise_dynamic_lds(ctx, (const void*)kernel, bytes, "context_create"); };
    raise(attention_tq_token_kernel<4, true, false>, token_lds<4>(kMaxWaves));
    raise(attention_tq_token_kernel<4, false, false>, token_lds<4>(kMaxWaves));
    raise(attention_tq_token_kernel<2, true, false>, token_lds<2>(kMaxWaves));
    raise(attention_tq_token_kernel<2, false, false>, token_lds<2>(kMaxWaves));
    raise(attention_tq_token_kernel<1, true, false>, token_lds<1>(kMaxWaves));
    raise(attention_tq_token_kernel<1, false, false>, token_lds<1>(kMaxWaves));
    raise(attention_tq_token_kernel<1, true, true>, token_lds<1>(kMaxWaves));
    raise(attention_tq_token_kernel<1, false, true>, token_lds<1>(kMaxWaves));
    return r;
}

namespace lh_attn {

bool prepare_rows_supported(const lh_context* ctx, uint32_t head_dim, uint32_t bits, uint32_t heads, uint32_t rows, bool own) {
    // Heads that have a CU each, or are one of a few there, are the shorter way with a workgroup each (four or eight waves instead of one).  Us, that form and this one:
    // queries alone of 256 dims up to four a CU (8 x 1 3.3 and 3.6; 8 x 64 3.9 and 3.5, but with the attention behind them, from partial tiles, 38.0 and 38.6; 8 x 200 so 69.3 and
    // 67.9), of 512 dims, whose four a workgroup share their pairs from three a CU on, up to there (8 x 64 36.7 and 37.7, 8 x 100 43.8 and 43.0; 5 x 180 alone 16.4 and 17.4);
    // with keys and values, whose chain of additions the others wait for, of 512 dims up to two a CU (10 x 1 6.7 and 8.4, 10 x 32 with product and attention 35.3 and 36.1, 10 x 64
    // 41.3 and 41.6, 10 x 100 49.6 and 48.5).
    const uint64_t all = (uint64_t)rows * heads, cus = (uint64_t)ctx->cu_count;
    return bits == 2 && heads <= kRowHeads && (head_dim == kDim || head_dim == 2 * kDim) &&
           all > (own ? (head_dim == kDim ? 0 : 2 * cus) : (head_dim == kDim || heads % 4 ? 4 : 3) * cus);
}

int launch_prepare_rows(lh_context* ctx, const char* op, const TokenPrep& t, uint32_t head_dim, uint32_t rows, float* rq, const float* levels, const uint32_t* positions, uint32_t position,
                        uint32_t ring_capacity, uint32_t lane_capacity, uint32_t q_heads, uint32_t kv_heads) {
    const RowsPrep r{rq, levels, positions, position, ring_capacity, lane_capacity, q_heads, kv_heads};
    const auto kernel = head_dim == kDim ? prepare_rows_kernel<4> : prepare_rows_kernel<8>;
    // As many heads a workgroup as leave every CU one.
    const uint32_t heads = q_heads + 2 * kv_heads, cus = (uint32_t)ctx->cu_count, each = (uint32_t)std::min<uint64_t>(((uint64_t)rows * heads + cus - 1) / cus, kRowHeads);
    const uint32_t groups = (heads + each - 1) / each, waves = (heads + groups - 1) / groups;
    hipLaunchKernelGGL(kernel, dim3(rows, groups), dim3(64 * waves), (size_t)waves * head_dim * 4, ctx->stream, r, t);
    return lh_check_launch(op);
}

bool short_supported(const lh_context* ctx, const AttnParams& p, uint64_t max_span) {
    static const bool off = [] { return getenv("LOCAL_HIP_ATTN_PAIR") != nullptr; }();      // (forces a form of the other kernel)
    // A CU for each workgroup, a wave for each group that a span may touch.  (One workgroup a query where the host knows the spans: see `more`.)
    return !off && p.head_dim == kDim && (uint64_t)p.num_queries * p.num_kv_heads * (p.mode == kBatched ? 2 : 1) <= (uint64_t)ctx->cu_count && (max_span + 62) / 64 + 1 <= kMaxWaves;
}

int launch_short(lh_context* ctx, const char* op, const AttnPointers& a, AttnParams& p, uint64_t max_span) {
    p.num_splits = 1;
    const uint32_t waves = std::max<uint32_t>(kHeads, (uint32_t)((max_span + 62) / 64 + 1)), queries = p.num_queries * p.num_kv_heads, cus = (uint32_t)ctx->cu_count;
    return queries * 4 <= cus ? launch<4>(ctx, op, a, p, waves) : queries * 2 <= cus ? launch<2>(ctx, op, a, p, waves) : launch<1>(ctx, op, a, p, waves);
}

// Waves for the groups that `positions` in a row may touch, one for each head at least.
static uint32_t group_waves(uint64_t positions) { return std::max<uint32_t>(kHeads, (uint32_t)((positions + 62) / 64 + 1)); }

bool token_supported(const lh_context* ctx, const AttnParams& p, const TokenPrep& t, uint64_t max_span) {
    if (max_span == 0 || !short_supported(ctx, p, max_span)) return false;
    if (t.k_codes && group_waves(max_span - 1) + 2 > kMaxWaves) return false;
    // The position's slot is written while the positions before it are read: on a ring it has to be none of theirs.
    const uint64_t most = p.mode != kBatched ? max_span : p.window ? p.window : p.ring_capacity ? UINT64_MAX : max_span;
    return !t.k_codes || p.ring_capacity == 0 || most <= p.ring_capacity;
}

int launch_token(lh_context* ctx, const char* op, const AttnPointers& a, AttnParams& p, const TokenPrep& t, uint64_t max_span) {
    p.num_splits = 1;
    const uint32_t waves = group_waves(t.k_codes ? max_span - 1 : max_span), queries = p.num_queries * p.num_kv_heads, cus = (uint32_t)ctx->cu_count;
    // A workgroup with all dims of a query can rotate its heads, which is worth the other dims' products in it: 64 lanes, window of 512, 14.5 us in one launch (14.2 on
    // another layer's cache) against 20.6 (18.3) for preparation, attention on four CUs a lane and rotation, two gaps not counted.
    if (t.rotated) return launch_token_form<1, true>(ctx, op, a, p, t, waves);
    return queries * 4 <= cus ? launch_token_form<4>(ctx, op, a, p, t, waves) : queries * 2 <= cus ? launch_token_form<2>(ctx, op, a, p, t, waves) : launch_token_form<1>(ctx, op, a, p, t, waves);
}

}  // namespace lh_attn
