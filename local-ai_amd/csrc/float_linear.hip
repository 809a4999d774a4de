// Products of activations with bf16 weights [N, K]:
//   linear_phased_kernel bf16 activations, K a multiple of 64, enough tiles of 128 x 128 for the chip: eight waves in two phases
//   linear_mfma_kernel   bf16 activations, K a multiple of 8: LDS-tiled bf16 MFMA 16x16x32, tiles loaded straight into LDS
//   linear_sliced_kernel the same where the tiles are few for the chip: small tiles, k shared out among a workgroup's waves
//   split_rows_kernel    f32 activations as three bf16 terms, for the three kernels above (the 32-bit runs)
//   linear_plain_kernel  everything else: f32 FMA on 64 x 64 tiles (ragged K, pieces that are not aligned)
//   matvec_bf16_kernel   one row, HBM-bound weight streaming, with the norm before the product done while x is staged
// All end in the same column segments (bias, activation, layout, residual add), and all but those for one row also run the experts of
// a mixture on the tiles of a routing plan.
#include "float_linear.hpp"
#include <algorithm>
#include <cstring>
#include <type_traits>

namespace {

typedef __attribute__((address_space(1))) const void gvoid;
typedef __attribute__((address_space(3))) void lvoid;

// 16 bytes per lane from global memory into LDS: lane i of the wave lands at lds + 16 i (`lds` wave-uniform).
__device__ __forceinline__ void load_lds16(const void* g, void* lds) {
    __builtin_amdgcn_global_load_lds((gvoid*)g, (lvoid*)lds, 16, 0, 0);
}

__device__ uint4 g_zero16 = {0u, 0u, 0u, 0u};   // what activation chunks past K read

// The rows this workgroup multiplies: tile `mt` of an ordinary product, or part `mt` of the tiles of an expert plan, whose rows are
// a multiple of bm.
struct RowTile { uint32_t begin, end, expert; };
__device__ __forceinline__ uint32_t row_tiles(const LhLinear& a, uint32_t bm) {
    return a.ex.tiles ? a.ex.n_tiles * (a.ex.tile_rows / bm) : (a.M + bm - 1) / bm;
}
__device__ __forceinline__ RowTile row_tile(const LhLinear& a, uint32_t mt, uint32_t bm) {
    if (a.ex.tiles == nullptr) return RowTile{mt * bm, min(mt * bm + bm, a.M), 0u};
    const uint32_t per = a.ex.tile_rows / bm;
    const uint32_t* t = a.ex.tiles + 3 * (mt / per);
    RowTile r{t[1], min(t[2], a.ex.slots), t[0]};
    if (r.expert >= a.ex.experts || r.begin >= r.end) return RowTile{0u, 0u, 0u};
    r.begin += mt % per * bm;
    r.end = min(r.end, r.begin + bm);
    return r;
}
__device__ __forceinline__ uint32_t a_row(const LhLinear& a, uint32_t slot) {
    if (!a.ex.gather) return slot;
    const uint32_t r = a.ex.slot_row[slot];
    return r < a.ex.rows ? r : 0u;
}
struct OutRow { uint32_t row; float weight; };
__device__ __forceinline__ OutRow out_row(const LhLinear& a, uint32_t slot) {
    OutRow o{slot, 1.0f};
    if (a.ex.tiles != nullptr) {
        if (a.ex.scatter) o.row = a.ex.slot_row[slot];
        if (a.ex.slot_weight) o.weight = a.ex.slot_weight[slot];
    }
    return o;
}

// Column and row tile of a workgroup: workgroups are dealt to the eight XCDs round robin, so each XCD gets a contiguous
// range of tiles (its L2 then sees the same weight panels again), walked in groups of four row tiles.
__device__ __forceinline__ void tile_of_block(uint32_t mt_n, uint32_t nt_n, uint32_t& mt, uint32_t& nt) {
    const uint32_t total = mt_n * nt_n, id = blockIdx.x;
    const uint32_t q = total >> 3, rem = total & 7, x = id & 7, i = id >> 3;
    const uint32_t t = (x < rem ? x * (q + 1) : rem * (q + 1) + (x - rem) * q) + i;
    const uint32_t gsz = 4 * nt_n, g = t / gsz, m_in = min(4u, mt_n - g * 4), r = t - g * gsz;
    mt = g * 4 + r % m_in;
    nt = r / m_in;
}

// Bias, activation and destination of columns n .. n + 3 (those below N) of one row of a product.
__device__ __forceinline__ void store4(const LhLinear& a, uint32_t slot, uint32_t n, const float4 acc, uint32_t pos0) {
    const OutRow o = out_row(a, slot);
    float v[4] = {acc.x, acc.y, acc.z, acc.w};
#pragma unroll
    for (int r = 0; r < 4; r++) v[r] = v[r] * o.weight + (a.bias && n + r < a.N ? a.bias[n + r] : 0.0f);
    const uint32_t s = lh_segment_of(a.seg, n);              // (of all four columns where the boundaries are aligned)
    if (a.seg.pairs) {
        if (a.seg.aligned4 && a.seg.act[s] == LH_ACT_SILU_PAIRS && !a.seg.f32[s]) {
            *reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(a.seg.out[s]) + (size_t)o.row * a.seg.ld[s] + (n - a.seg.n0[s]) / 2) =
                lh_pack_bf(v[0] * lh_sigmoid(v[0]) * v[1], v[2] * lh_sigmoid(v[2]) * v[3]);
            return;
        }
        lh_segment_store_pair(a.seg, o.row, n, v[0], v[1], pos0);   // every count of columns is even here
        if (n + 2 < a.N) lh_segment_store_pair(a.seg, o.row, n + 2, v[2], v[3], pos0);
        return;
    }
    if (!a.seg.aligned4 || !a.seg.vec4[s]) {
#pragma unroll 1
        for (uint32_t r = 0; r < 4 && n + r < a.N; r++) lh_segment_store(a.seg, o.row, n + r, r == 0 ? v[0] : r == 1 ? v[1] : r == 2 ? v[2] : v[3], pos0);
        return;
    }
    const uint32_t p = lh_segment_at_position(a.seg, s) ? pos0 + o.row : o.row;
    if (p >= a.seg.rows[s]) return;
    uint32_t c = n - a.seg.n0[s];
    if (a.seg.head[s] != a.seg.padded[s]) { const uint32_t h = c / a.seg.head[s]; c = h * a.seg.padded[s] + (c - h * a.seg.head[s]); }
    const size_t idx = (size_t)p * a.seg.ld[s] + c;
    const uint32_t act = a.seg.act[s];
    if (act != LH_ACT_NONE) {
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] = lh_activate(v[r], act);
    }
    if (a.seg.f32[s]) {
        float4* d = reinterpret_cast<float4*>(static_cast<float*>(a.seg.out[s]) + idx);
        float4 t = make_float4(v[0], v[1], v[2], v[3]);
        if (a.seg.accumulate) { const float4 x = *d; t.x += x.x; t.y += x.y; t.z += x.z; t.w += x.w; }
        *d = t;
    } else {
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.seg.out[s]) + idx) = make_uint2(lh_pack_bf(v[0], v[1]), lh_pack_bf(v[2], v[3]));
    }
}

// Place of four-column piece c of row m in a wave's tile of N columns in LDS.
template <int N> __device__ __forceinline__ uint32_t piece(uint32_t m, uint32_t c) { return m * (N / 4) + (c ^ (m & (N / 4 < 8 ? N / 4 - 1 : 7))); }

// A wave's finished tile of N columns into a value cache: four lanes store the quarters of a block of 32 positions of one column,
// 16 bytes each where the tile has all of a quarter.
template <int N>
__device__ __forceinline__ void store_blocks(const LhLinear& a, uint32_t s, const float* tile, const RowTile& rt, uint32_t n0, uint32_t pos0, uint32_t lane) {
    const uint32_t first = pos0 + rt.begin, last = min(pos0 + rt.end, a.seg.rows[s]), b0 = first >> 5;      // positions [first, last)
    if (first >= last) return;
    const uint32_t blocks = ((last - 1) >> 5) - b0 + 1, g = lane & 3;
#pragma unroll 1
    for (uint32_t j = lane >> 2; j < N && n0 + j < a.N; j += 16) {
        uint32_t c = n0 + j - a.seg.n0[s];
        if (a.seg.head[s] != a.seg.padded[s]) { const uint32_t h = c / a.seg.head[s]; c = h * a.seg.padded[s] + (c - h * a.seg.head[s]); }
        uint16_t* d = static_cast<uint16_t*>(a.seg.out[s]) + ((size_t)b0 * a.seg.ld[s] + c) * 32 + g * 8;
        const float bias = a.bias ? a.bias[n0 + j] : 0.0f;
#pragma unroll 1
        for (uint32_t b = b0; b < b0 + blocks; b++, d += (size_t)a.seg.ld[s] * 32) {
            uint16_t v[8];
            bool all = true, in[8];
#pragma unroll
            for (uint32_t i = 0; i < 8; i++) {                // entries 8 g + i: positions 4 g + i and 16 + 4 g + i - 4
                const uint32_t p = b * 32 + (i >> 2) * 16 + g * 4 + (i & 3);
                in[i] = p >= first && p < last;
                all = all && in[i];
                const uint32_t m = in[i] ? p - first : 0u;
                v[i] = lh_f2bf(lh_activate(tile[piece<N>(m, j >> 2) * 4 + (j & 3)] + bias, a.seg.act[s]));
            }
            if (all) *reinterpret_cast<uint4*>(d) = make_uint4(v[0] | (uint32_t)v[1] << 16, v[2] | (uint32_t)v[3] << 16, v[4] | (uint32_t)v[5] << 16, v[6] | (uint32_t)v[7] << 16);
            else {
#pragma unroll
                for (uint32_t i = 0; i < 8; i++) if (in[i]) d[i] = v[i];
            }
        }
    }
}

// A wave's finished tile of M x N from LDS to its destination.
template <int M, int N>
__device__ __forceinline__ void store_tile(const LhLinear& a, const float4* tile, const RowTile& rt, uint32_t n0, uint32_t pos0, uint32_t lane) {
    const uint32_t s = lh_segment_of(a.seg, n0);
    if (a.seg.layout[s] == LH_BLOCKS_AT_POSITION && !a.seg.f32[s] && s == lh_segment_of(a.seg, min(n0 + N, a.N) - 1) && a.ex.tiles == nullptr) {
        store_blocks<N>(a, s, reinterpret_cast<const float*>(tile), rt, n0, pos0, lane);
        return;
    }
#pragma unroll 1
    for (uint32_t e = lane; e < M * N / 4; e += 64) {
        const uint32_t m = e / (N / 4), c = e % (N / 4), n = n0 + c * 4, slot = rt.begin + m;
        if (slot >= rt.end || n >= a.N) continue;
        store4(a, slot, n, tile[piece<N>(m, c)], pos0);
    }
}

// What is left to do for the tile of TI * 16 rows and TJ * 16 columns that a wave has in registers (column 4 TJ (lane >> 4) + 4 j + t
// of row lane & 15 in register t of acc[i][j]: the kernels deal the rows of W to the matrix instructions that way).  A lane finishes
// its 4 TJ neighbouring columns in registers and stores them in 16-byte pieces.  Value blocks, and segments that are not made of
// multiples of 4 TJ, go through LDS, `box`, which is the wave's own.  (All through LDS, in pieces of four columns with their
// segments looked up one by one: 93 us instead of 60 for the product of 2048 x 2048 x 8192 with gelu.)
enum { kThroughLds = -1, kNoActivation = 0, kGelu, kSilu, kSiluPairs, kReluSquared };   // kSilu, kReluSquared: of the segments that have it

// Where a lane's columns go, the same for all its rows.
struct LaneColumns {
    uint32_t n, s, c, ld, act, f32, at_position, rows;         // first column, its segment and its place there
    char* out;                                                // of row 0
    __device__ __forceinline__ LaneColumns(const LhSegments& seg, uint32_t first) : n(first), s(lh_segment_of(seg, first)) {
        c = n - seg.n0[s];
        act = seg.act[s]; f32 = seg.f32[s]; ld = seg.ld[s]; rows = seg.rows[s];
        if (act == LH_ACT_SILU_PAIRS) c >>= 1;
        else if (seg.head[s] != seg.padded[s]) { const uint32_t h = c / seg.head[s]; c = h * seg.padded[s] + (c - h * seg.head[s]); }
        at_position = lh_segment_at_position(seg, s);
        out = static_cast<char*>(seg.out[s]) + (size_t)c * (f32 ? 4 : 2);
    }
};
// v / (1 + exp(-z)) as a division and expf have it, from a quarter of v and of -z (a denominator past 2^126 has no reciprocal): the
// hardware's exponential of t = -z log2 e, with what the rounding of t leaves (-z - t ln 2; the nearest f32 to ln 2 is good to 3e-9) put
// back, and a quotient corrected once; v_div_fixup has the infinities, NaN and exponentials past f32.  For 2048 x 2048 x 8192 with gelu
// 62.5 us, with expf and a division 68, with exp2 and a reciprocal alone 60.5.  Of 4.2 million bf16 results with silu not the nearest: 47, 56
// and 66 (whose error grows with |z|: up to 15 x 2^-24 seen behind a pair, 7 expected of f32 arithmetic).
__device__ __forceinline__ float over_one_plus_exp(float v_4, float minus_z_4) {
    const float m = __builtin_amdgcn_fmed3f(minus_z_4, -100.0f, INFINITY), t = 5.7707801635558536f * m, p = __builtin_amdgcn_exp2f(t);
    const float whole = __builtin_fmaf(p, 0.25f, 0.25f), d = __builtin_fmaf(p, __builtin_fmaf(t, -0.17328679513998632f, m), whole);
    const float r = __builtin_amdgcn_rcpf(d), q = v_4 * r;
    return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-d, q, v_4), r, q), whole, v_4);
}
__device__ __forceinline__ float silu_column(float v) { return over_one_plus_exp(0.25f * v, -0.25f * v); }
template <int EPI> __device__ __forceinline__ float activate_columns(float v, uint32_t act) {
    if constexpr (EPI == kGelu) return over_one_plus_exp(0.25f * v, -0.3989422804014327f * (v + 0.044715f * v * v * v));
    if constexpr (EPI == kSilu) return act == LH_ACT_SILU ? silu_column(v) : v;
    if constexpr (EPI == kReluSquared) { const float r = fmaxf(v, 0.0f); return act == LH_ACT_RELU_SQUARED ? r * r : v; }
    return v;
}
template <int EPI, int TI, int TJ>
__device__ __forceinline__ void store_columns(const LhLinear& a, const lh_f32x4 (*acc)[TJ], const LaneColumns& col, uint32_t slot0, uint32_t end, uint32_t pos0) {
    constexpr int CN = 4 * TJ;
    if (col.n >= a.N) return;
    float bias[CN];
#pragma unroll
    for (int j = 0; j < CN; j++) bias[j] = a.bias ? a.bias[col.n + j] : 0.0f;
    // A row's destination; what is there already is requested a row ahead.
    struct Row { uint32_t p; float weight; bool valid; };
    auto row = [&](int i) {
        const uint32_t slot = slot0 + i * 16;
        Row r{0, 1.0f, slot < end};
        if (r.valid) {
            const OutRow o = out_row(a, slot);
            r.p = col.at_position ? pos0 + o.row : o.row; r.weight = o.weight;
            r.valid = r.p < col.rows;
        }
        return r;
    };
    const bool add = EPI == kNoActivation && a.seg.accumulate && col.f32;
    float4 x[2][TJ];
    auto fetch = [&](const Row& r, float4 (&d)[TJ]) {
        if (!add || !r.valid) return;
#pragma unroll
        for (int j = 0; j < TJ; j++) d[j] = reinterpret_cast<const float4*>(col.out + (size_t)r.p * col.ld * 4)[j];
    };
    Row next = row(0);
    fetch(next, x[0]);
#pragma unroll
    for (int i = 0; i < TI; i++) {
        const Row r = next;
        if (i + 1 < TI) { next = row(i + 1); fetch(next, x[(i + 1) & 1]); }
        if (!r.valid) continue;
        float v[CN];
#pragma unroll
        for (int j = 0; j < CN; j++) v[j] = activate_columns<EPI>(acc[i][j >> 2][j & 3] * r.weight + bias[j], col.act);
        if (EPI != kSiluPairs && col.f32) {
            float4* d = reinterpret_cast<float4*>(col.out + (size_t)r.p * col.ld * 4);
            if (add) {
#pragma unroll
                for (int j = 0; j < TJ; j++) { const float4 y = x[i & 1][j]; v[4 * j] += y.x; v[4 * j + 1] += y.y; v[4 * j + 2] += y.z; v[4 * j + 3] += y.w; }
            }
#pragma unroll
            for (int j = 0; j < TJ; j++) d[j] = make_float4(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]);
            continue;
        }
        constexpr int W = EPI == kSiluPairs ? TJ : 2 * TJ;     // words of two bf16
        uint32_t w[W];
#pragma unroll
        for (int j = 0; j < W; j++) {
            if constexpr (EPI == kSiluPairs) w[j] = lh_pack_bf(silu_column(v[4 * j]) * v[4 * j + 1], silu_column(v[4 * j + 2]) * v[4 * j + 3]);
            else w[j] = lh_pack_bf(v[2 * j], v[2 * j + 1]);
        }
        char* d = col.out + (size_t)r.p * col.ld * 2;
        if constexpr (W == 8) { reinterpret_cast<uint4*>(d)[0] = make_uint4(w[0], w[1], w[2], w[3]); reinterpret_cast<uint4*>(d)[1] = make_uint4(w[4], w[5], w[6], w[7]); }
        else if constexpr (W == 4) *reinterpret_cast<uint4*>(d) = make_uint4(w[0], w[1], w[2], w[3]);
        else if constexpr (W == 2) *reinterpret_cast<uint2*>(d) = make_uint2(w[0], w[1]);
        else *reinterpret_cast<uint32_t*>(d) = w[0];
    }
}

// The same into a value cache, for whole blocks of 32 positions.  Four neighbouring lanes have positions 4 q .. 4 q + 3 of four
// columns; transposed among themselves, over the two 16-row tiles of a block, each has the 16 bytes 4 g .. of one column's block.
__device__ __forceinline__ void transpose_quads(uint32_t (&u)[4], uint32_t lane) {
    const bool odd = lane & 1, high = lane & 2;
#pragma unroll
    for (int e = 0; e < 4; e += 2) {                          // 2 x 2 blocks
        const uint32_t give = odd ? u[e] : u[e + 1], got = (uint32_t)lh_dpp_i<LH_DPP_QUAD_XOR1>((int)give);
        if (odd) u[e] = got; else u[e + 1] = got;
    }
#pragma unroll
    for (int e = 0; e < 2; e++) {
        const uint32_t give = high ? u[e] : u[e + 2], got = (uint32_t)lh_dpp_i<LH_DPP_QUAD_XOR2>((int)give);
        if (high) u[e] = got; else u[e + 2] = got;
    }
}
template <int EPI, int TI, int TJ>
__device__ __forceinline__ void store_whole_blocks(const LhLinear& a, const lh_f32x4 (*acc)[TJ], const LaneColumns& col, uint32_t position, uint32_t lane) {
    const uint32_t q = (lane >> 2) & 3, k = lane & 3;
    uint16_t* out = reinterpret_cast<uint16_t*>(a.seg.out[col.s]) + ((size_t)(position >> 5) * col.ld + col.c + k) * 32 + q * 8;
#pragma unroll
    for (int j = 0; j < TJ; j++) {
        float bias[4];
#pragma unroll
        for (int t = 0; t < 4; t++) bias[t] = a.bias ? a.bias[col.n + 4 * j + t] : 0.0f;
#pragma unroll
        for (int b = 0; b < TI / 2; b++) {
            uint32_t u[4];
#pragma unroll
            for (int t = 0; t < 4; t++) u[t] = lh_pack_bf(activate_columns<EPI>(acc[2 * b][j][t] + bias[t], col.act), activate_columns<EPI>(acc[2 * b + 1][j][t] + bias[t], col.act));
            transpose_quads(u, lane);
            *reinterpret_cast<uint4*>(out + ((size_t)b * col.ld + 4 * j) * 32) =
                make_uint4(__builtin_amdgcn_perm(u[1], u[0], 0x05040100u), __builtin_amdgcn_perm(u[3], u[2], 0x05040100u),
                           __builtin_amdgcn_perm(u[1], u[0], 0x07060302u), __builtin_amdgcn_perm(u[3], u[2], 0x07060302u));
        }
    }
}

template <int EPI, int TI, int TJ>
__device__ __forceinline__ void finish_tile(const LhLinear& a, const lh_f32x4 (*acc)[TJ], const RowTile& rt, uint32_t row0, uint32_t nw, uint32_t lane, float4* box) {
    if (nw >= a.N) return;
    const uint32_t pos0 = a.seg.position ? *a.seg.position : 0u, g = lane >> 4;
    if constexpr (EPI != kThroughLds) {
        const uint32_t s0 = lh_segment_of(a.seg, nw), s1 = lh_segment_of(a.seg, min(nw + 16 * TJ, a.N) - 1), first = rt.begin + row0, at = pos0 + first;
        bool blocks = false;                                  // in any of the segments: the wave's columns may hold a whole one between two others
#pragma unroll
        for (uint32_t s = 0; s < 4; s++) blocks = blocks || (s >= s0 && s <= s1 && a.seg.layout[s] == LH_BLOCKS_AT_POSITION);
        if (!blocks) {
            store_columns<EPI, TI, TJ>(a, acc, LaneColumns(a.seg, nw + g * 4 * TJ), first + (lane & 15), rt.end, pos0);
            return;
        }
        if constexpr (EPI != kSiluPairs && TI % 2 == 0) {
            if (blocks && s0 == s1 && !a.seg.f32[s0] && nw + 16 * TJ <= a.N && at % 32 == 0 && first + TI * 16 <= rt.end && at + TI * 16 <= a.seg.rows[s0] && a.ex.tiles == nullptr) {
                store_whole_blocks<EPI, TI, TJ>(a, acc, LaneColumns(a.seg, nw + g * 4 * TJ), at, lane);
                return;
            }
        }
    }
    constexpr int RP = TI < 4 ? TI : 4;                       // 16-row tiles at a time
#pragma unroll
    for (int h = 0; h < TI / RP; h++) {
#pragma unroll
        for (int i = 0; i < RP; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++) {
                const lh_f32x4 v = acc[h * RP + i][j];
                box[piece<16 * TJ>(i * 16 + (lane & 15), g * TJ + j)] = make_float4(v[0], v[1], v[2], v[3]);
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        const uint32_t b = rt.begin + row0 + h * RP * 16;
        if (b < rt.end) store_tile<RP * 16, 16 * TJ>(a, box, RowTile{b, min(b + RP * 16, rt.end), rt.expert}, nw, pos0, lane);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
}

// Rows of W in the order in which the lanes 0 .. 15 of tile j take them, and the chunk permutation under which eight neighbouring
// lanes read different banks.
template <int TJ> __device__ __forceinline__ uint32_t dealt_row(uint32_t lane, uint32_t j) { return ((lane & 15) >> 2) * 4 * TJ + j * 4 + (lane & 3); }
template <int TJ> __device__ __forceinline__ uint32_t dealt_swizzle(uint32_t row) { return (row & 3) | (row / (4 * TJ) & 1) << 2; }

// ---- matrix cores ------------------------------------------------------------------------------------------------------
// 256 threads, 2 x 2 waves of BM/2 x BN/2 outputs.  A k step is 64 wide: a tile row is eight 16-byte chunks, chunk c of row r
// kept at place c ^ (r & 7) of its row so that the fragment reads of sixteen rows fall on different banks (the loads
// write LDS in order, so the permutation is applied to their global addresses).  NS buffers, one barrier per step: step kt is
// multiplied while the loads of the NS - 1 steps after it are on their way.
// The weights are the MFMA's row operand: lane = output row (lane & 15), four output columns per tile.
template <int N> __device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory"); }

template <int BM, int BN, int NS, int EPI>
__global__ __launch_bounds__(256) void linear_mfma_kernel(const LhLinear a) {
    constexpr int TI = BM / 32, TJ = BN / 32, CA = BM / 32, CB = BN / 32;
    static_assert(NS * (BM + BN) * 128 >= BM * BN * 4, "the output tile must fit the staging buffers");
    __shared__ uint4 sm[NS][(BM + BN) * 8];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave >> 1, wn = wave & 1;
    uint32_t mt, nt;
    tile_of_block(row_tiles(a, BM), (a.N + BN - 1) / BN, mt, nt);
    const RowTile rt = row_tile(a, mt, BM);
    if (rt.begin >= rt.end) return;
    const uint32_t n0 = nt * BN, K = a.K, steps = (K + 63) / 64, nk = steps * a.parts;
    const uint16_t* A = static_cast<const uint16_t*>(a.A);
    const uint16_t* W = a.W + (size_t)rt.expert * a.N * K;

    const uint16_t* pa[CA];
    const uint16_t* pb[CB];
    // the chunk this thread brings in, of every row it serves
    const uint32_t src = (tid & 7) ^ ((tid >> 3) & 7), src_b = (tid & 7) ^ dealt_swizzle<TJ>(tid >> 3);
#pragma unroll
    for (int i = 0; i < CA; i++) {
        const uint32_t r = min(rt.begin + i * 32 + (tid >> 3), rt.end - 1);
        pa[i] = A + (size_t)a_row(a, r) * a.lda + src * 8;
    }
#pragma unroll
    for (int i = 0; i < CB; i++) pb[i] = W + (size_t)min(n0 + i * 32 + (tid >> 3), a.N - 1) * K + src_b * 8;

    auto load_step = [&](int buf, uint32_t step) {
        uint4* base = &sm[buf][wave * 64];
        const uint32_t part = (step >= steps) + (step >= 2 * steps), kt = step - part * steps;
        const size_t ka = (size_t)part * a.part_stride + kt * 64;
        if (kt * 64 + 64 <= K) {
#pragma unroll
            for (int i = 0; i < CA; i++) load_lds16(pa[i] + ka, base + i * 256);
#pragma unroll
            for (int i = 0; i < CB; i++) load_lds16(pb[i] + kt * 64, base + (CA + i) * 256);
        } else {                                             // the last step of a ragged K: chunks past it read zeros
            const bool past = kt * 64 + src * 8 >= K, past_b = kt * 64 + src_b * 8 >= K;
#pragma unroll
            for (int i = 0; i < CA; i++) load_lds16(past ? (const void*)&g_zero16 : (const void*)(pa[i] + ka), base + i * 256);
#pragma unroll
            for (int i = 0; i < CB; i++) load_lds16(past_b ? (const void*)&g_zero16 : (const void*)(pb[i] + kt * 64), base + (CA + i) * 256);
        }
    };

    lh_f32x4 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++) acc[i][j] = (lh_f32x4){0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int i = 0; i < NS - 1; i++) if (i < (int)nk) load_step(i, i);
    uint32_t buf = 0;
    for (uint32_t kt = 0; kt < nk; kt++) {
        if (kt + NS - 1 <= nk) wait_loads<(NS - 2) * (CA + CB)>();   // step kt has arrived; the later steps may still be coming
        else wait_loads<0>();
        lh_lds_barrier();
        if (kt + NS - 1 < nk) load_step(buf == 0 ? NS - 1 : buf - 1, kt + NS - 1);
        const uint4* as = sm[buf];
        buf = buf + 1 == NS ? 0 : buf + 1;
        const uint4* bs = as + BM * 8;
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            lh_bf16x8 fa[TI], fb[TJ];
            const uint32_t c = ks * 4 + (lane >> 4);
#pragma unroll
            for (int i = 0; i < TI; i++) {
                const uint32_t r = wm * (BM / 2) + i * 16 + (lane & 15);
                fa[i] = __builtin_bit_cast(lh_bf16x8, as[r * 8 + (c ^ (r & 7))]);
            }
#pragma unroll
            for (int j = 0; j < TJ; j++) {
                const uint32_t r = wn * (BN / 2) + dealt_row<TJ>(lane, j);
                fb[j] = __builtin_bit_cast(lh_bf16x8, bs[r * 8 + (c ^ (lane & 7))]);
            }
#pragma unroll
            for (int i = 0; i < TI; i++)
#pragma unroll
                for (int j = 0; j < TJ; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);
        }
    }

    __syncthreads();
    finish_tile<EPI, TI, TJ>(a, acc, rt, wm * (BM / 2), n0 + wn * (BN / 2), lane, reinterpret_cast<float4*>(&sm[0][0]) + wave * (BM * BN / 16));
}

// Few tiles for the chip: what bounds a product then is how much of it is on its way to a CU (16 KB a step and three steps ahead in the
// kernel above: a step takes as long as a third of a trip to memory).  Here every wave multiplies the whole tile over a slice of k,
// the steps wave, wave + W, ..., out of buffers of its own in LDS, all NS of them requested ahead, with no barrier until the W sums meet
// at the end, in one order.  A buffer is requested again as soon as its fragments are in registers.
template <int BM, int BN, int W, int NS, int EPI>
__global__ __launch_bounds__(64 * W) void linear_sliced_kernel(const LhLinear a) {
    constexpr int TI = BM / 16, TJ = BN / 16, CA = BM / 8, CB = BN / 8, STEP = (BM + BN) * 8, PER = CA + CB;
    static_assert((NS - 1) * PER < 64, "requests are counted in six bits");
    static_assert(NS * STEP * 16 >= BM * BN * 4 + 2048, "a wave's sums and its part of the output tile must fit its buffers");
    extern __shared__ uint4 sm[];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t mt, nt;
    tile_of_block(row_tiles(a, BM), (a.N + BN - 1) / BN, mt, nt);
    const RowTile rt = row_tile(a, mt, BM);
    if (rt.begin >= rt.end) return;
    const uint32_t n0 = nt * BN, K = a.K, steps = (K + 63) / 64, nk = steps * a.parts;
    const uint16_t* A = static_cast<const uint16_t*>(a.A);
    const uint16_t* Wt = a.W + (size_t)rt.expert * a.N * K;

    const uint16_t *pa[CA], *pb[CB];
    const uint32_t src = (lane & 7) ^ (lane >> 3);
#pragma unroll
    for (int i = 0; i < CA; i++) pa[i] = A + (size_t)a_row(a, min(rt.begin + i * 8 + (lane >> 3), rt.end - 1)) * a.lda + src * 8;
#pragma unroll
    for (int i = 0; i < CB; i++) pb[i] = Wt + (size_t)min(n0 + i * 8 + (lane >> 3), a.N - 1) * K + src * 8;

    uint4* const ring = sm + wave * NS * STEP;
    auto load_step = [&](uint32_t buf, uint32_t step) {
        uint4* base = ring + buf * STEP;
        const uint32_t part = (step >= steps) + (step >= 2 * steps), kt = step - part * steps;
        const size_t ka = (size_t)part * a.part_stride + kt * 64;
        if (kt * 64 + 64 <= K) {
#pragma unroll
            for (int i = 0; i < CA; i++) load_lds16(pa[i] + ka, base + i * 64);
#pragma unroll
            for (int i = 0; i < CB; i++) load_lds16(pb[i] + kt * 64, base + (CA + i) * 64);
        } else {                                             // the last step of a ragged K: chunks past it read zeros
            const bool past = kt * 64 + src * 8 >= K;
#pragma unroll
            for (int i = 0; i < CA; i++) load_lds16(past ? (const void*)&g_zero16 : (const void*)(pa[i] + ka), base + i * 64);
#pragma unroll
            for (int i = 0; i < CB; i++) load_lds16(past ? (const void*)&g_zero16 : (const void*)(pb[i] + kt * 64), base + (CA + i) * 64);
        }
    };

    lh_f32x4 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++) acc[i][j] = (lh_f32x4){0.f, 0.f, 0.f, 0.f};

    const uint32_t mine = nk > wave ? (nk - wave + W - 1) / W : 0;
#pragma unroll
    for (int i = 0; i < NS; i++) if (i < (int)mine) load_step(i, wave + i * W);
    uint32_t buf = 0;
    const uint32_t g = lane >> 4, at[2] = {g ^ (lane & 7), (g + 4) ^ (lane & 7)};
    for (uint32_t i = 0; i < mine; i++) {
        if (i + NS <= mine) wait_loads<(NS - 1) * PER>();     // step i has arrived; the later steps may still be coming
        else wait_loads<0>();
        const uint4 *as = ring + buf * STEP + (lane & 15) * 8, *bs = as + BM * 8;
        lh_bf16x8 fa[2][TI], fb[2][TJ];
#pragma unroll
        for (int s = 0; s < 2; s++) {
#pragma unroll
            for (int t = 0; t < TI; t++) fa[s][t] = __builtin_bit_cast(lh_bf16x8, as[t * 128 + at[s]]);
#pragma unroll
            for (int t = 0; t < TJ; t++) fb[s][t] = __builtin_bit_cast(lh_bf16x8, bs[t * 128 + at[s]]);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (i + NS < mine) load_step(buf, wave + (i + NS) * W);
        buf = buf + 1 == NS ? 0 : buf + 1;
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int t = 0; t < TI; t++)
#pragma unroll
                for (int u = 0; u < TJ; u++) acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[s][u], fa[s][t], acc[t][u], 0, 0, 0);
    }

    // Every wave's sums to LDS; a wave then finishes tiles of 32 x 16.
    lh_f32x4* const sums = reinterpret_cast<lh_f32x4*>(sm);
    __syncthreads();
#pragma unroll
    for (int t = 0; t < TI; t++)
#pragma unroll
        for (int u = 0; u < TJ; u++) sums[(wave * TI * TJ + t * TJ + u) * 64 + lane] = acc[t][u];
    __syncthreads();
    float4* const box = reinterpret_cast<float4*>(sums + W * TI * TJ * 64) + wave * 128;
#pragma unroll 1
    for (uint32_t e = wave; e < TI / 2 * TJ; e += W) {
        const uint32_t t = e / TJ * 2, u = e % TJ;
        lh_f32x4 sum[2][1];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const lh_f32x4* from = sums + ((t + h) * TJ + u) * 64 + lane;
            sum[h][0] = from[0];
#pragma unroll
            for (int w = 1; w < W; w++) sum[h][0] += from[w * TI * TJ * 64];
        }
        finish_tile<EPI, 2, 1>(a, sum, rt, t * 16, n0 + u * 16, lane, box);
    }
}

// Large products, K a multiple of 64.  Eight waves in two groups of four, one wave of either group on each SIMD, half a period
// apart: while one group multiplies, the other fetches its next fragments from LDS and requests tiles, so that the matrix cores of
// a SIMD always have one wave's work (2140 cycles per step of 64 on a 256 x 256 tile, of which 2048 are matrix-core cycles; with all
// waves in the same phase: 3100).  A phase ends in a barrier that all waves pass; a wave waits for its own requests, counted, before
// the barrier behind which they are read.  Tiles per step and buffers:
//   256 x 256  waves of 128 x 64, two buffers of 64 KB, refilled in two parts as soon as both groups have read a part
//   256 x 128  waves of 64 x 64, three buffers of 48 KB
//   128 x 128  waves of 64 x 64; the groups take the even and the odd steps, five buffers of 32 KB (with four, requests were half a
//              period later: 81 us instead of 74 at 2048 x 8192 x 2048 with weights from HBM), and their sums meet at the end
// Rows and chunks as in linear_mfma_kernel.
__device__ __forceinline__ void phase_end() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
// The fragments asked for in this phase are here, and all but the last N requested pieces.
template <int N> __device__ __forceinline__ void read_end() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// Whether the tiles are an expert plan's is known when the kernel is compiled: asked at run time it cost every plain product 0.9 us before the first
// load (1500 x 3072 x 2048 27.0 -> 27.9 us).
template <int BM, int BN, int EPI, bool PLAN>
__global__ __launch_bounds__(512) void linear_phased_kernel(const LhLinear a) {
    constexpr bool kWide = BN == 256, kHalves = BM == 128;               // (256 x 128 is neither)
    constexpr int TI = kWide ? 8 : 4, SLOT = (BM + BN) * 8;              // 16-row tiles of a wave; 16-byte pieces of a buffer
    constexpr int T = kHalves ? 256 : 512, CA = BM * 8 / T, CB = BN * 8 / T;
    extern __shared__ uint4 sm[];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), group = wave >> 2;
    const uint32_t wm = kWide ? group : kHalves ? (wave >> 1) & 1 : wave >> 1, wn = kWide ? wave & 3 : wave & 1;
    uint32_t mt, nt;
    tile_of_block(PLAN ? row_tiles(a, BM) : (a.M + BM - 1) / BM, (a.N + BN - 1) / BN, mt, nt);
    const RowTile rt = PLAN ? row_tile(a, mt, BM) : RowTile{mt * BM, min(mt * BM + BM, a.M), 0u};
    if (PLAN && rt.begin >= rt.end) return;
    const uint32_t n0 = nt * BN, K = a.K, steps = K / 64, nk = steps * a.parts;
    const char* A = static_cast<const char*>(a.A);
    const char* W = reinterpret_cast<const char*>(PLAN ? a.W + (size_t)rt.expert * a.N * K : a.W);

    const uint32_t lt = kHalves ? tid & 255 : tid, src = ((lt & 7) ^ ((lt >> 3) & 7)) * 16, src_b = ((lt & 7) ^ dealt_swizzle<4>(lt >> 3)) * 16;
    uint32_t pa[CA], pb[CB];                                   // byte offsets: the host has checked that they fit
#pragma unroll
    for (int i = 0; i < CA; i++) {
        const uint32_t row = min(rt.begin + i * (T / 8) + (lt >> 3), rt.end - 1);
        pa[i] = (PLAN ? a_row(a, row) : row) * a.lda * 2 + src;
    }
#pragma unroll
    for (int i = 0; i < CB; i++) pb[i] = min(n0 + i * (T / 8) + (lt >> 3), a.N - 1) * K * 2 + src_b;
    uint4* const to = sm + (kHalves ? wave & 3 : wave) * 64;
    auto part_of = [&](uint32_t kt) { return (uint32_t)(kt >= steps) + (kt >= 2 * steps); };
    auto load_a = [&](uint32_t buf, uint32_t kt, int i) {
        const uint32_t part = part_of(kt);
        load_lds16(A + (size_t)part * a.part_stride * 2 + (kt - part * steps) * 128 + pa[i], to + buf * SLOT + i * T);
    };
    auto load_b = [&](uint32_t buf, uint32_t kt, int i) { load_lds16(W + (kt - part_of(kt) * steps) * 128 + pb[i], to + buf * SLOT + BM * 8 + i * T); };
    auto load_step = [&](uint32_t buf, uint32_t kt) {
#pragma unroll
        for (int i = 0; i < CA; i++) load_a(buf, kt, i);
#pragma unroll
        for (int i = 0; i < CB; i++) load_b(buf, kt, i);
    };

    lh_f32x4 acc[TI][4];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = (lh_f32x4){0.f, 0.f, 0.f, 0.f};
    const uint32_t g = lane >> 4, at[2] = {g ^ (lane & 7), (g + 4) ^ (lane & 7)};
    const uint4 *ra = sm + (wm * TI * 16 + (lane & 15)) * 8, *rb = sm + (BM + wn * 64 + dealt_row<4>(lane, 0)) * 8;
    lh_bf16x8 fa[2][4], fb[2][4];
    auto read_a = [&](uint32_t buf, int h) {
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int i = 0; i < 4; i++) fa[s][i] = __builtin_bit_cast(lh_bf16x8, ra[buf * SLOT + (h * 4 + i) * 128 + at[s]]);
    };
    auto read_b = [&](uint32_t buf) {
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int j = 0; j < 4; j++) fb[s][j] = __builtin_bit_cast(lh_bf16x8, rb[buf * SLOT + j * 32 + at[s]]);
    };
    auto multiply = [&](int h) {                              // 64 x 64 outputs over 64 columns of k, the wave ahead of the one that reads
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[h * 4 + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[s][j], fa[s][i], acc[h * 4 + i][j], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
    };

    if constexpr (kWide) {
        // Part one of a buffer: B and the rows that the waves multiply first (0 .. 63 of either half); part two: the other rows.
        auto part1 = [&](uint32_t kt) { for (int i = 0; i < 4; i++) load_b(kt & 1, kt, i); load_a(kt & 1, kt, 0); load_a(kt & 1, kt, 2); };
        auto part2 = [&](uint32_t kt) { load_a(kt & 1, kt, 1); load_a(kt & 1, kt, 3); };
        part1(0); part2(0);
        if (nk > 1) { part1(1); read_end<8>(); } else read_end<2>();
        if (group) phase_end();
        uint32_t kt = 0;
        for (; kt + 2 < nk; kt++) {
            read_b(kt & 1); read_a(kt & 1, 0); part2(kt + 1); read_end<8>();
            multiply(0); phase_end();
            read_a(kt & 1, 1); part1(kt + 2); read_end<8>();
            multiply(1); phase_end();
        }
        if (kt + 1 < nk) {
            read_b(kt & 1); read_a(kt & 1, 0); part2(kt + 1); read_end<8>();
            multiply(0); phase_end();
            read_a(kt & 1, 1); read_end<2>();
            multiply(1); phase_end();
            kt++;
        }
        read_b(kt & 1); read_a(kt & 1, 0); read_end<0>();
        multiply(0); phase_end();
        read_a(kt & 1, 1); read_end<0>();
        multiply(1); phase_end();
    } else if constexpr (kHalves) {
        // A group's steps are kt = group, group + 2, ...  Step kt is in buffer kt mod 5; while a group reads step kt it requests its step
        // kt + 4: step kt - 1, which was there, has been read by the other group.
        const uint32_t mine = (nk + 1 - group) / 2, most = (nk + 1) / 2;
        if (mine > 0) load_step(group, group);
        if (mine > 1) { load_step(group + 2, group + 2); wait_loads<8>(); } else wait_loads<0>();
        phase_end();
        if (group) phase_end();
        uint32_t kt = group, buf = group;
        for (uint32_t i = 0; i < most; i++) {
            if (i + 2 < mine) load_step(buf == 0 ? 4 : buf - 1, kt + 4);
            if (i < mine) { read_a(buf, 0); read_b(buf); }
            read_end<63>();
            if (i < mine) multiply(0);
            if (i + 2 < mine) wait_loads<8>(); else wait_loads<0>();
            phase_end();
            kt += 2;
            buf = buf >= 3 ? buf - 3 : buf + 2;
        }
    } else {
        // Step kt is in buffer kt mod 3; a wave requests step kt + 2 while it reads step kt: step kt - 1, which was there, has been
        // read by both groups.
        load_step(0, 0);
        if (nk > 1) { load_step(1, 1); read_end<6>(); } else read_end<0>();
        if (group) phase_end();
        uint32_t buf = 0, kt = 0;
        for (; kt + 2 < nk; kt++) {
            read_a(buf, 0); read_b(buf); load_step(buf == 0 ? 2 : buf - 1, kt + 2);
            buf = buf == 2 ? 0 : buf + 1;
            read_end<6>();
            multiply(0); phase_end();
        }
        for (; kt < nk; kt++) {
            read_a(buf, 0); read_b(buf);
            buf = buf == 2 ? 0 : buf + 1;
            read_end<0>();
            multiply(0); phase_end();
        }
    }
    if (!group) phase_end();

    uint32_t row0 = wm * TI * 16;
    if constexpr (kHalves) {                                  // group 0 finishes the upper 32 rows of a wave's tile, group 1 the lower
        lh_f32x4* const box = reinterpret_cast<lh_f32x4*>(sm) + (wave & 3) * 512 + lane;
#pragma unroll
        for (int e = 0; e < 8; e++) box[group * 2048 + e * 64] = group ? acc[e >> 2][e & 3] : acc[2 + (e >> 2)][e & 3];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const lh_f32x4 other = box[(group ^ 1) * 2048 + e * 64];
            acc[e >> 2][e & 3] = group ? other + acc[2 + (e >> 2)][e & 3] : acc[e >> 2][e & 3] + other;
        }
        row0 += group * 32;
        __syncthreads();
    }
    finish_tile<EPI, kHalves ? 2 : TI, 4>(a, acc, rt, row0, n0 + wn * 64, lane, reinterpret_cast<float4*>(sm) + wave * 1024);
}

// ---- f32 rows as bf16 terms ----------------------------------------------------------------------------------------------
// An f32 value is the sum of three bf16 values that are cut off, not rounded, so that all have its sign: 8 bits each, 24 in all.  The
// products with bf16 weights are then exact and summed in f32, as FMA has them, on the matrix cores; a row becomes its lowest terms,
// its middle terms and its leading terms, one after the other.  No term is zero, or an infinite weight would give NaN where it gives an
// infinity times the value itself: a value of fewer bits passes its last one on to the terms below (values from 2^-110 up; smaller ones
// lose bits below bf16's range).
// (The products of a pass over 333 rows at width 1024: 184 us on average on the FMA units, 30 and 4.5 for the terms.)
__global__ __launch_bounds__(256) void split_rows_kernel(const float* __restrict__ x, uint16_t* __restrict__ out, uint32_t rows, uint32_t K, uint32_t lda, uint32_t stride) {
    const uint32_t row = blockIdx.y * 4 + threadIdx.x / 64;
    if (row >= rows) return;
    for (uint32_t k = (blockIdx.x * 64 + (threadIdx.x & 63)) * 4; k < stride; k += gridDim.x * 256) {
        const float4 v = k < K ? *reinterpret_cast<const float4*>(x + (size_t)row * lda + k) : make_float4(0.f, 0.f, 0.f, 0.f);
        const float f[4] = {v.x, v.y, v.z, v.w};
        uint32_t t[3][4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t u = __builtin_bit_cast(uint32_t, f[j]);
            if ((u & 0x7F800000u) == 0x7F800000u) {           // infinite, or no number (which stays none when it is cut off)
                t[0][j] = t[1][j] = t[2][j] = (u >> 16) | ((u & 0x007FFFFFu) ? 0x40u : 0u);
                continue;
            }
            const float hi = __builtin_bit_cast(float, u & 0xFFFF0000u), r = f[j] - hi;
            // (the last bit of a bf16 value: seven places below its exponent, none where that is below the normal ones)
            auto bit_of = [](float v, uint32_t places) {
                const uint32_t e = __builtin_bit_cast(uint32_t, v) & 0x7F800000u, s = __builtin_bit_cast(uint32_t, v) & 0x80000000u;
                return e > (places << 23) ? __builtin_bit_cast(float, (e - (places << 23)) | s) : 0.0f;
            };
            float top = hi, mid = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, r) & 0xFFFF0000u), low = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, r - mid) & 0xFFFF0000u);
            if (r == 0.0f) { mid = low = bit_of(hi, 8); top = hi - (mid + low); }
            else if (r == mid) { low = bit_of(mid, 7); mid -= low; }
            t[0][j] = __builtin_bit_cast(uint32_t, low) >> 16;
            t[1][j] = __builtin_bit_cast(uint32_t, mid) >> 16;
            t[2][j] = __builtin_bit_cast(uint32_t, top) >> 16;
        }
        uint16_t* o = out + (size_t)row * 3 * stride + k;
#pragma unroll
        for (int z = 0; z < 3; z++) *reinterpret_cast<uint2*>(o + (size_t)z * stride) = make_uint2(t[z][0] | t[z][1] << 16, t[z][2] | t[z][3] << 16);
    }
}

// Workgroups for 256 columns each where that makes up to six a CU, for 1024 beyond.  Few are bound by a lane's trips to memory, one behind the other; many by how
// they begin and end.  (With a product of 64 columns: 333 x 1024 12.7 us with four trips, 11.0 with one, 333 x 4096 27.8 and 27.2; 1000 x 2048 19.8 and 21.2, 2048 x 2048 21.9 and
// 25.7, 4096 x 1024 18.5 and 21.5.)
uint32_t split_grid(uint32_t rows, uint32_t stride, uint64_t cus) {
    const uint32_t groups = (stride + 255) / 256;
    return (uint64_t)groups * ((rows + 3) / 4) <= 6 * cus ? groups : (stride + 1023) / 1024;
}

// ---- f32 FMA -----------------------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void linear_plain_kernel(const LhLinear a) {
    constexpr int BK = 16;
    __shared__ float as[BK][64 + 4], bs[BK][64 + 4];
    const uint32_t tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    const uint32_t nt_n = (a.N + 63) / 64, mt = blockIdx.x / nt_n, nt = blockIdx.x % nt_n;
    const RowTile rt = row_tile(a, mt, 64);
    if (rt.begin >= rt.end) return;
    const T* A = static_cast<const T*>(a.A);
    const uint16_t* W = a.W + (size_t)rt.expert * a.N * a.K;
    const uint32_t n0 = nt * 64, K = a.K, pos0 = a.seg.position ? *a.seg.position : 0u;
    float acc[4][4] = {};
    for (uint32_t k0 = 0; k0 < K; k0 += BK) {
        for (uint32_t e = tid; e < 64 * BK; e += 256) {
            const uint32_t r = e >> 4, k = k0 + (e & 15);
            const bool ka = k < K;
            as[e & 15][r] = ka && rt.begin + r < rt.end ? lh_ld(A, (size_t)a_row(a, rt.begin + r) * a.lda + k) : 0.0f;
            bs[e & 15][r] = ka && n0 + r < a.N ? lh_bf2f(W[(size_t)(n0 + r) * K + k]) : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < BK; k++) {
            float x[4], w[4];
#pragma unroll
            for (int i = 0; i < 4; i++) { x[i] = as[k][ty * 4 + i]; w[i] = bs[k][tx * 4 + i]; }
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] = __builtin_fmaf(x[i], w[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t slot = rt.begin + ty * 4 + i;
        if (slot >= rt.end) continue;
        const OutRow o = out_row(a, slot);
        if (a.seg.pairs) {                                // (an expert's weight and a bias do not occur with pairs of a plain product)
#pragma unroll
            for (int j = 0; j < 4; j += 2) {
                const uint32_t n = n0 + tx * 4 + j;
                if (n < a.N) lh_segment_store_pair(a.seg, o.row, n, acc[i][j] + (a.bias ? a.bias[n] : 0.0f), acc[i][j + 1] + (a.bias ? a.bias[n + 1] : 0.0f), pos0);
            }
            continue;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t n = n0 + tx * 4 + j;
            if (n < a.N) lh_segment_store(a.seg, o.row, n, acc[i][j] * o.weight + (a.bias ? a.bias[n] : 0.0f), pos0);
        }
    }
}

// ---- one row -----------------------------------------------------------------------------------------------------------
// Place of element k in the staged vector: the two halves of an 8-element chunk lie in planes of 64 x 16 bytes, so that the
// 16-byte reads of a wave (lane = chunk) are in order.
__device__ __forceinline__ uint32_t x_place(uint32_t k) {
    const uint32_t chunk = k >> 3, j = k & 7;
    return (((chunk >> 6) * 2 + (j >> 2)) << 8) + ((chunk & 63) << 2) + (j & 3);
}

template <int STAGE>
__device__ void stage_vector(const VectorStage& st, float* xs, float* scratch, uint32_t K) {
    auto gate = [&](uint32_t k) { return lh_gate(st.gate_f32 ? static_cast<const float*>(st.gate)[k] : lh_bf2f(static_cast<const uint16_t*>(st.gate)[k]), st.gate_act); };
    auto value = [&](uint32_t k) {
        if constexpr (STAGE == kPlain) return st.x_f32 ? static_cast<const float*>(st.x)[k] : lh_bf2f(static_cast<const uint16_t*>(st.x)[k]);
        float v = static_cast<const float*>(st.x)[k];
        if (STAGE == kNorm && st.add) v += st.add[k];
        if constexpr (STAGE == kGated) if (st.gate_first) v *= gate(k);
        return v;
    };
    auto weight = [&](uint32_t k) {
        const float w = STAGE != kGated || st.norm_weight ? st.norm_weight[k] : 1.0f;
        if constexpr (STAGE == kGated) return st.gate_first ? w : w * gate(k);
        return w;
    };
    const uint32_t padded = (K + 511) / 512 * 512;
    if constexpr (STAGE == kResidual) {
        float s = 0.0f;
        for (uint32_t k = threadIdx.x; k < K; k += blockDim.x) { const float y = st.add[k]; s += y * y; }
        const float r = rsqrtf(lh_block_sum(s, scratch) / (float)K + st.eps);
        for (uint32_t k = threadIdx.x; k < padded; k += blockDim.x) {
            const float v = k < K ? __builtin_fmaf(st.add[k] * st.norm_weight[k], r, value(k)) : 0.0f;
            xs[x_place(k)] = v;
            if (st.store && blockIdx.x == 0 && k < K) st.store[k] = v;
        }
    } else if constexpr (STAGE == kPlain) {
        for (uint32_t k = threadIdx.x; k < padded; k += blockDim.x) xs[x_place(k)] = k < K ? value(k) : 0.0f;
    } else {
        constexpr int R = 8;                                  // elements a thread keeps between the passes; the rest are read again
        float keep[R], wk[R];
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < R; i++) {
            const uint32_t k = threadIdx.x + i * blockDim.x;
            keep[i] = k < K ? value(k) : 0.0f;
            wk[i] = k < K ? weight(k) : 0.0f;
            s += keep[i] * keep[i];
        }
        for (uint32_t k = threadIdx.x + R * blockDim.x; k < K; k += blockDim.x) { const float v = value(k); s += v * v; }
        const float r = rsqrtf(lh_block_sum(s, scratch) / (float)K + st.eps);
        const bool store = STAGE == kNorm && st.store != nullptr && blockIdx.x == 0;
#pragma unroll
        for (int i = 0; i < R; i++) {
            const uint32_t k = threadIdx.x + i * blockDim.x;
            if (k < padded) xs[x_place(k)] = keep[i] * r * wk[i];
            if (store && k < K) st.store[k] = keep[i];
        }
        for (uint32_t k = threadIdx.x + R * blockDim.x; k < padded; k += blockDim.x) {
            float v = 0.0f, w = 0.0f;
            if (k < K) {
                v = value(k);
                w = weight(k);
                if (store) st.store[k] = v;
            }
            xs[x_place(k)] = v * r * w;
        }
    }
    __syncthreads();
}

// Which rows a wave (or workgroup) takes: every `count`-th from `first` on; of (gate, up) pairs both.
struct RowWalk {
    const uint32_t first, count, pairs;
    __device__ __forceinline__ uint32_t row(uint32_t i) const { return pairs ? 2 * (first + (i >> 1) * count) + (i & 1) : first + i * count; }
    __device__ __forceinline__ uint32_t rows(uint32_t N) const {  // how many of N
        const uint32_t n = pairs ? N / 2 : N, r = first < n ? (n - first - 1) / count + 1 : 0u;
        return pairs ? 2 * r : r;
    }
};

// Stores the finished sums of rows i0 .. i0 + n - 1 of a walk, one per lane.
__device__ __forceinline__ void store_sums(const LhSegments& seg, const float* bias, const RowWalk& walk, uint32_t i0, uint32_t n, uint32_t lane, float v) {
    const uint32_t row = walk.row(i0 + lane);
    if (bias && lane < n) v += bias[row];
    if (seg.cap != 0.0f) v = seg.cap * tanhf(v / seg.cap);
    if (walk.pairs) {                                         // n is even, and a pair's factors are in neighbouring lanes
        const float up = lh_dpp_f<LH_DPP_QUAD_XOR1>(v);
        if (lane < n && !(lane & 1)) lh_segment_put(seg, 0, row >> 1, v * lh_sigmoid(v) * up);
    } else if (lane < n) lh_segment_store(seg, 0, row, v, seg.position ? *seg.position : 0u);
}

// The finished sums of a wave's rows, one per lane, stored 64 at a time: bias, activation and destination then cost one pass
// for all of them, and no load of that pass has to wait for weights that were requested in between.
struct RowSums {
    const LhSegments& seg;
    const float* bias;
    const RowWalk& walk;
    const uint32_t lane;
    uint32_t i0 = 0, n = 0;
    float mine = 0.0f, before = 0.0f;
    bool known = false;
    // What the first 64 sums are added to is requested ahead of the products, where it is one plain row of values.
    __device__ __forceinline__ void request(uint32_t rows) {
        known = seg.accumulate && seg.count == 1 && !seg.pairs && !lh_segment_at_position(seg, 0) && seg.head[0] == seg.padded[0];
        if (known && lane < rows) before = static_cast<const float*>(seg.out[0])[walk.row(lane)];
    }
    __device__ __forceinline__ void keep(float total) { mine = n++ == lane ? total : mine; }      // up to 64 of them, then a flush
    __device__ __forceinline__ void add(float total) {
        keep(total);
        if (n == 64) flush();
    }
    __device__ __forceinline__ void flush() {
        if (known && i0 == 0) {
            const uint32_t row = walk.row(lane);
            if (lane < n) static_cast<float*>(seg.out[0])[row] = before + lh_activate(bias ? mine + bias[row] : mine, seg.act[0]);
        } else store_sums(seg, bias, walk, i0, n, lane, mine);
        i0 += n;
        n = 0;
    }
};

// A wave takes rows round robin over the grid, 8 weights (16 bytes) per lane and load, NL loads per pass of a row; the loads
// of the next pass are issued before the arithmetic of the current one.  Past the row's end the address is clamped and the
// staged vector is zero.  VEC false (K not a multiple of 8): single weights.
template <int STAGE, int NL, bool VEC>
__global__ __launch_bounds__(256) void matvec_bf16_kernel(const VectorStage st, const uint16_t* __restrict__ W, const float* __restrict__ bias, const LhSegments seg,
                                                         uint32_t N, uint32_t K) {
    extern __shared__ __align__(16) float xs[];
    __shared__ float scratch[4];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    stage_vector<STAGE>(st, xs, scratch, K);
    const RowWalk walk{blockIdx.x * 4 + wave, gridDim.x * 4, seg.pairs};
    RowSums sums{seg, bias, walk, lane};
    if constexpr (VEC) {
        constexpr uint32_t kPass = 512u * NL;
        const uint32_t ppr = (K + kPass - 1) / kPass, last = (K >> 3) - 1;
        uint32_t at = 0, row = walk.row(0), pass = 0;
        auto issue = [&](uint4 (&v)[NL], uint32_t r, uint32_t ps) {
            const uint16_t* wr = W + (size_t)r * K;
#pragma unroll
            for (int c = 0; c < NL; c++) v[c] = lh_ld16_stream(wr + 8 * min(ps * (kPass >> 3) + 64u * c + lane, last));
        };
        float acc = 0.0f;
        auto consume = [&](const uint4 (&v)[NL], uint32_t r, uint32_t ps) {
#pragma unroll
            for (int c = 0; c < NL; c++) {
                const uint32_t q = ps * NL + c;
                if (q * 512 >= K) break;
                const float4 x0 = *reinterpret_cast<const float4*>(&xs[(q * 2) * 256 + lane * 4]), x1 = *reinterpret_cast<const float4*>(&xs[(q * 2 + 1) * 256 + lane * 4]);
                const float xv[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
                const uint32_t wv[4] = {v[c].x, v[c].y, v[c].z, v[c].w};
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    acc = __builtin_fmaf(__builtin_bit_cast(float, wv[j] << 16), xv[2 * j], acc);
                    acc = __builtin_fmaf(__builtin_bit_cast(float, wv[j] & 0xFFFF0000u), xv[2 * j + 1], acc);
                }
            }
            if (ps + 1 == ppr) { sums.add(lh_group_sum(acc, 64)); acc = 0.0f; }
        };
        auto step = [&](const uint4 (&cur)[NL], uint4 (&nxt)[NL]) {   // false: that was the wave's last pass
            uint32_t nrow = row, npass = pass + 1;
            if (npass == ppr) { npass = 0; nrow = walk.row(++at); }
            const bool more = nrow < N;
            if (more) issue(nxt, nrow, npass);
            consume(cur, row, pass);
            row = nrow; pass = npass;
            return more;
        };
        uint4 p[NL], q[NL];
        if (row < N) {
            issue(p, row, 0);
            while (step(p, q) && step(q, p)) {}
        }
    } else {
        for (uint32_t i = 0, row; (row = walk.row(i)) < N; i++) {
            float acc = 0.0f;
            for (uint32_t k = lane; k < K; k += 64) acc = __builtin_fmaf(lh_bf2f(W[(size_t)row * K + k]), xs[x_place(k)], acc);
            sums.add(lh_group_sum(acc, 64));
        }
    }
    sums.flush();
}

// The same with the vector in registers (K up to 512 * NL), which the waves of a workgroup bring in together; the weights of two rows are
// requested right behind it and every wait leaves the younger loads on their way.  What bounds it is the length of one such chain, not
// the bytes.  (Four waves, each with the vector for itself and one row ahead: 10.0 us a launch on average over the products of a step
// behind a norm, 2048 columns and 2048 to 32000 rows, 10.6 behind a gate, 5.9 with neither; with eight waves 8.9, 5.8 and 4.0.)
// COPY: one plain row of values, which also goes to `copy` (memory of the host, as a rule); the sums of a workgroup meet in LDS and leave in
// runs of a row a wave, 32 bytes, not in single words.  (32000 x 2048 22.4 us, 21.8 without; a copy over the bus behind it took 4.7 and the step to it.)
template <int STAGE, int NL, int WAVES, bool COPY = false>
__global__ __launch_bounds__(64 * WAVES) void matvec_bf16_reg_kernel(const VectorStage st, const uint16_t* __restrict__ W, const float* __restrict__ bias, const LhSegments seg,
                                                             uint32_t N, uint32_t K, float* __restrict__ copy) {
    __shared__ LhVectorSpace<WAVES> space;
    __shared__ float results[COPY ? WAVES : 1][65];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), last = (K >> 3) - 1;
    const RowWalk walk{blockIdx.x * WAVES + wave, gridDim.x * WAVES, seg.pairs};
    const uint32_t rows = walk.rows(N);
    struct Row { uint4 w[NL]; } v[2];
    auto issue = [&](Row& x, uint32_t i) {
        const uint16_t* wr = W + (size_t)min(walk.row(i), N - 1) * K;
#pragma unroll
        for (int c = 0; c < NL; c++) x.w[c] = lh_ld16_stream(wr + 8 * min(64u * c + lane, last));
    };
    LhSharedVector<STAGE, NL, WAVES> x;
    x.fetch(st, K, lane, wave);
    lh_first_rows(v, max(rows, 1u), [&](Row& r, uint32_t i) { issue(r, rows ? i : 0u); });
    RowSums sums{seg, bias, walk, lane};
    float xr[NL][8];
    x.finish(st, K, lane, wave, blockIdx.x == 0 && st.store != nullptr, space, xr);
    if (!COPY && rows == 0) return;
    if constexpr (!COPY) sums.request(rows);
    lh_walk_rows(v, rows, issue, [&](const Row& r, uint32_t) {
        float acc = 0.0f;
#pragma unroll
        for (int c = 0; c < NL; c++) acc = lh_dot8(r.w[c], xr[c], acc);
        sums.keep(lh_group_sum(acc, 64));
    });
    if constexpr (COPY) {
        results[wave][lane] = sums.mine;                      // rows: at most 64 a wave
        lh_lds_barrier();
        const uint32_t row = walk.first - wave + threadIdx.x % WAVES + threadIdx.x / WAVES * walk.count;
        if (row >= N) return;
        float v = results[threadIdx.x % WAVES][threadIdx.x / WAVES];
        if (bias) v += bias[row];
        if (seg.cap != 0.0f) v = seg.cap * tanhf(v / seg.cap);
        static_cast<float*>(seg.out[0])[row] = v;
        copy[row] = v;
    } else sums.flush();
}

// Rows longer than a wave's registers: the eight waves of a workgroup take an eighth of the columns each, and the parts of up to 64
// rows, all that a workgroup takes, meet in LDS, where wave 0 adds them.  Plain vectors only: a norm would need all parts.  (Four waves with a
// quarter each and one row ahead: 9.6 us for 2048 x 8192; now 7.8.)
template <int NL, int R>
__global__ __launch_bounds__(512) void matvec_bf16_part_kernel(const VectorStage st, const uint16_t* __restrict__ W, const float* __restrict__ bias, const LhSegments seg,
                                                              uint32_t N, uint32_t K, uint32_t part) {
    __shared__ float sums[kVectorWaves][64];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), k0 = wave * part, len = k0 < K ? min(part, K - k0) : 0u;   // part: a multiple of 8
    const uint32_t last = len ? (len >> 3) - 1 : 0u, kb = len ? k0 : 0u;
    const RowWalk walk{blockIdx.x, gridDim.x, seg.pairs};
    const uint32_t rows = walk.rows(N);
    if (rows == 0) return;
    struct Row { uint4 w[NL]; } v[R];
    auto issue = [&](Row& x, uint32_t i) {
        const uint16_t* wr = W + (size_t)walk.row(i) * K + kb;
#pragma unroll
        for (int c = 0; c < NL; c++) x.w[c] = lh_ld16_stream(wr + 8 * min(64u * c + lane, last));
    };
    LhEither8 raw[NL];                                        // the vector first (see LhSharedVector)
#pragma unroll
    for (int c = 0; c < NL; c++) raw[c].load(st.x, st.x_f32, kb + 8 * min(64u * c + lane, last));
    lh_first_rows(v, rows, issue);
    RowSums total{seg, bias, walk, lane};
    float xr[NL][8], mine = 0.0f;
#pragma unroll
    for (int c = 0; c < NL; c++) {
        raw[c].get(st.x_f32, xr[c]);
#pragma unroll
        for (int j = 0; j < 8; j++) xr[c][j] = (64u * c + lane) * 8 < len ? xr[c][j] : 0.0f;
    }
    if (wave == 0) total.request(rows);
    lh_walk_rows(v, rows, issue, [&](const Row& x, uint32_t i) {
        float acc = 0.0f;
#pragma unroll
        for (int c = 0; c < NL; c++) acc = lh_dot8(x.w[c], xr[c], acc);
        acc = lh_group_sum(acc, 64);
        mine = i == lane ? acc : mine;
    });
    sums[wave][lane] = mine;
    lh_lds_barrier();
    if (wave != 0) return;
    float t = 0.0f;
#pragma unroll
    for (int w = 0; w < kVectorWaves; w++) t += sums[w][lane];
    total.mine = t; total.n = rows;
    total.flush();
}

// A workgroup for every CU first; a second one where rows are short and each of its waves still has two (32000 x 1024: 11.9 us
// against 12.5; 8192 x 2048: 7.8 against 7.65).  A wave's sums (`each`) fit its lanes.
uint32_t one_row_grid(uint64_t takes, uint32_t K, uint32_t waves, uint32_t each, uint64_t cus) {
    const uint64_t most = std::max(cus, K <= 1024 ? std::min<uint64_t>(2 * cus, (takes + 15) / 16) : 0);
    return (uint32_t)std::max<uint64_t>(std::min<uint64_t>((takes + waves - 1) / waves, most), (takes + waves * each - 1) / (waves * each));
}

// Results that also go to pinned memory: by the product's own launch, in pieces of 32 bytes, as long as the product is what takes the time.  Many results of
// short rows are bound by the bus, where a copy behind the product is faster (us for the host, so and with the copy: 1024 columns, 32000 rows 28 and 30,
// 65536 45 and 45, 262144 153 and 149; 256 columns 24 and 26, 34 and 34, 105 and 98; 1536 columns, 128000 rows 92 and 94).
bool copied_in_product(uint32_t K, uint32_t N) { return K <= 2048 && (K > 1024 || N <= 65536); }

constexpr uint32_t kMaxVectorK = 36864;   // 144 KB of staged f32 activations

template <int STAGE>
int launch_vector(lh_context* ctx, const VectorStage& st, const uint16_t* W, const float* bias, const LhSegments& seg, uint32_t N, uint32_t K, const char* op,
                  float* copy = nullptr) {
    // `copy` of the one plain f32 row of results: by the launch itself, or by one behind it.
    const auto copied = [&]() {
        const int r = lh_check_launch(op);
        if (r != LH_OK || !copy) return r;
        lh_launch_copy_out(ctx->stream, seg.out[0], copy, (size_t)N * 4);
        return lh_check_launch(op);
    };
    LH_REQUIRE(K > 0 && K <= kMaxVectorK, "%s: k %u outside 1..=%u", op, K, kMaxVectorK);
    const size_t lds = (size_t)(K + 511) / 512 * 512 * 4;
    const uint32_t takes = seg.pairs ? N / 2 : N;             // rows, or pairs of rows
    const bool vec = K % 8 == 0 && ((uintptr_t)W & 15) == 0;
    const uint64_t cus = (uint64_t)ctx->cu_count;
    // Up to eight rows per CU: workgroups of four waves, so that twice as many CUs have one (2048 x 2048 behind a norm 4.7 us with eight,
    // 4.1 with four, 1024 x 2048 4.3 and 3.7, 512 x 512 3.1 and 2.8), and beyond 2048 columns, for plain vectors, a row over eight waves
    // (below: 1024 x 4096 5.2 us and 4.4, 2048 x 4096 6.4 and 5.6; 4096 x 4096 7.5 and 7.8).
    const bool few = takes <= 8 * cus;
    if (vec && K <= 4096 && lh_stage_aligned(st) && !(STAGE == kPlain && K > 2048 && few)) {
        const uint32_t w = K <= 2048 && few ? 4 : kVectorWaves;
        const uint32_t grid = one_row_grid(takes, K, w, seg.pairs ? 32 : 64, cus);
#define LH_MVC(NLOADS, WAVES, COPY) hipLaunchKernelGGL((matvec_bf16_reg_kernel<STAGE, NLOADS, WAVES, COPY>), dim3(grid), dim3(64 * WAVES), 0, ctx->stream, st, W, bias, seg, N, K, copy)
#define LH_MVR(NLOADS, WAVES) LH_MVC(NLOADS, WAVES, false)
        if constexpr (STAGE == kNorm) if (copy && w == 8 && copied_in_product(K, N)) {
            if (K <= 512) LH_MVC(1, 8, true);
            else if (K <= 1024) LH_MVC(2, 8, true);
            else LH_MVC(4, 8, true);
            return lh_check_launch(op);
        }
        if (w == 4) {
            if (K <= 512) LH_MVR(1, 4);
            else if (K <= 1024) LH_MVR(2, 4);
            else LH_MVR(4, 4);
        } else if (K <= 512) LH_MVR(1, 8);
        else if (K <= 1024) LH_MVR(2, 8);
        else if (K <= 2048) LH_MVR(4, 8);
        else LH_MVR(8, 8);
#undef LH_MVR
#undef LH_MVC
        return copied();
    }
    if constexpr (STAGE == kPlain) if (vec && K <= 16384 && lh_stage_aligned(st)) {
        const uint32_t part = ((K + 7) / 8 + 7) / 8 * 8, each = seg.pairs ? 32 : 64;
        const uint32_t grid = (uint32_t)std::max<uint64_t>(std::min<uint64_t>(takes, cus), ((uint64_t)takes + each - 1) / each);
        if (part <= 512) hipLaunchKernelGGL((matvec_bf16_part_kernel<1, 4>), dim3(grid), dim3(64 * kVectorWaves), 0, ctx->stream, st, W, bias, seg, N, K, part);
        else if (part <= 1024) hipLaunchKernelGGL((matvec_bf16_part_kernel<2, 4>), dim3(grid), dim3(64 * kVectorWaves), 0, ctx->stream, st, W, bias, seg, N, K, part);
        else hipLaunchKernelGGL((matvec_bf16_part_kernel<4, 2>), dim3(grid), dim3(64 * kVectorWaves), 0, ctx->stream, st, W, bias, seg, N, K, part);
        return copied();
    }
    const uint32_t grid = (uint32_t)std::min<uint64_t>(((uint64_t)takes + 3) / 4, (uint64_t)ctx->cu_count * 4);
#define LH_MV(NLOADS, V)                                                                                                               \
    do {                                                                                                                               \
        if (lds > 64 * 1024 - 64) {                                                                                                    \
            const int rr = lh_raise_dynamic_lds(ctx, (const void*)matvec_bf16_kernel<STAGE, NLOADS, V>, lds, op);                      \
            if (rr != LH_OK) return rr;                                                                                                \
        }                                                                                                                              \
        hipLaunchKernelGGL((matvec_bf16_kernel<STAGE, NLOADS, V>), dim3(grid), dim3(256), lds, ctx->stream, st, W, bias, seg, N, K);    \
    } while (0)
    if (!vec) LH_MV(1, false);
    else if (K <= 512) LH_MV(1, true);
    else if (K <= 1024) LH_MV(2, true);
    else LH_MV(4, true);
#undef LH_MV
    return copied();
}

int check_common(lh_batch* batch, const lh_buffer* weight, const lh_buffer* bias, uint32_t k, uint64_t n, const char* op) {
    LH_REQUIRE(k > 0, "%s: k is 0", op);
    LH_NEED(weight, (size_t)n * k * 2, op, "weight");
    if (bias) LH_NEED(bias, (size_t)n * 4, op, "bias");
    return LH_OK;
}
#define LH_TRY(expr)                  \
    do {                              \
        const int rt__ = (expr);      \
        if (rt__ != LH_OK) return rt__; \
    } while (0)

int vector_entry(lh_batch* batch, const char* op, int stage, const VectorStage& st, const lh_buffer* weight, const lh_buffer* bias, uint32_t k,
                 uint32_t count, const uint32_t* ns, const uint32_t* acts, const uint32_t* heads, const uint32_t* padded, const uint32_t* layouts,
                 lh_buffer* const* outputs, int output_dtype, int accumulate, const lh_buffer* position, float cap = 0.0f, lh_buffer* copy = nullptr) {
    LhSegments seg;
    LH_TRY(lh_make_segments(seg, op, 1, 0, count, ns, acts, heads, padded, layouts, outputs, output_dtype, accumulate, position));
    seg.cap = cap;
    LH_REQUIRE(!seg.pairs || seg.count == 1, "%s: pairs beside other segments", op);
    const uint32_t n = seg.n0[seg.count];
    LH_TRY(check_common(batch, weight, bias, k, n, op));
    const uint16_t* W = (const uint16_t*)weight->ptr;
    const float* b = bias ? (const float*)bias->ptr : nullptr;
    int r;
    if (stage == kResidual) r = launch_vector<kResidual>(batch->ctx, st, W, b, seg, n, k, op);
    else if (stage == kPlain) r = launch_vector<kPlain>(batch->ctx, st, W, b, seg, n, k, op);
    else if (stage == kNorm) r = launch_vector<kNorm>(batch->ctx, st, W, b, seg, n, k, op, copy ? static_cast<float*>(copy->ptr) : nullptr);
    else r = launch_vector<kGated>(batch->ctx, st, W, b, seg, n, k, op);
    if (r == LH_OK) batch->dispatch_count++;
    return r;
}

}  // namespace

// Rows of an expert plan's tiles: a kernel takes them in parts, so they are the largest part that can be of use.
uint32_t lh_expert_tile_rows(uint32_t slots, uint32_t experts) {
    const uint32_t each = slots / (experts ? experts : 1);
    return each >= 192 ? 256u : each >= 128 ? 128u : 64u;
}

// Whether a lane can finish `per_lane` neighbouring columns by itself, and which activations it then meets.
static int epilogue_of(const LhSegments& seg, uint32_t per_lane) {
    bool none = true, gelu = true, silu = true, pairs = true, relu = true;
    for (uint32_t s = 0; s < seg.count; s++) {
        const uint32_t act = seg.act[s], size = seg.f32[s] ? 4 : 2;
        if (seg.n0[s] % per_lane || seg.n0[s + 1] % per_lane || (act != LH_ACT_NONE && seg.f32[s])) return kThroughLds;
        if (seg.head[s] != seg.padded[s] && seg.head[s] % per_lane) return kThroughLds;
        if (((uintptr_t)seg.out[s] | (uintptr_t)seg.ld[s] * size | (uintptr_t)seg.padded[s] * size) & 15) return kThroughLds;
        none = none && act == LH_ACT_NONE;
        gelu = gelu && act == LH_ACT_GELU_TANH;
        silu = silu && (act == LH_ACT_NONE || act == LH_ACT_SILU);
        relu = relu && (act == LH_ACT_NONE || act == LH_ACT_RELU_SQUARED);
        pairs = pairs && act == LH_ACT_SILU_PAIRS;
    }
    if (seg.accumulate && !none) return kThroughLds;
    return none ? kNoActivation : gelu ? kGelu : silu ? kSilu : relu ? kReluSquared : pairs ? kSiluPairs : kThroughLds;
}

template <class Launch>
static void with_epilogue(int epilogue, Launch launch) {
    switch (epilogue) {
        case kNoActivation: launch(std::integral_constant<int, kNoActivation>()); break;
        case kGelu: launch(std::integral_constant<int, kGelu>()); break;
        case kSilu: launch(std::integral_constant<int, kSilu>()); break;
        case kSiluPairs: launch(std::integral_constant<int, kSiluPairs>()); break;
        case kReluSquared: launch(std::integral_constant<int, kReluSquared>()); break;
        default: launch(std::integral_constant<int, kThroughLds>());
    }
}
template <int BM, int BN, int NS>
static int launch_mfma(lh_context* ctx, const LhLinear& a, uint64_t grid, const char* op) {
    LH_REQUIRE(grid < 0x7FFFFFFFull, "%s: %u x %u outputs", op, a.M, a.N);
    if (grid == 0) return LH_OK;
    with_epilogue(epilogue_of(a.seg, BN / 8), [&](auto epi) {
        hipLaunchKernelGGL((linear_mfma_kernel<BM, BN, NS, decltype(epi)::value>), dim3((uint32_t)grid), dim3(256), 0, ctx->stream, a);
    });
    return lh_check_launch(op);
}
template <int BM, int BN, int NS>
static int launch_sliced(lh_context* ctx, const LhLinear& a, uint64_t grid, const char* op) {
    LH_REQUIRE(grid < 0x7FFFFFFFull, "%s: %u x %u outputs", op, a.M, a.N);
    if (grid == 0) return LH_OK;
    constexpr size_t lds = (size_t)4 * NS * (BM + BN) * 128;
    int r = LH_OK;
    with_epilogue(epilogue_of(a.seg, 4), [&](auto epi) {
        const auto kernel = linear_sliced_kernel<BM, BN, 4, NS, decltype(epi)::value>;
        r = lh_raise_dynamic_lds(ctx, (const void*)kernel, lds, op);
        if (r == LH_OK) hipLaunchKernelGGL(kernel, dim3((uint32_t)grid), dim3(256), lds, ctx->stream, a);
    });
    return r == LH_OK ? lh_check_launch(op) : r;
}
template <int BM, int BN>
static int launch_phased(lh_context* ctx, const LhLinear& a, uint64_t grid, const char* op) {
    LH_REQUIRE(grid < 0x7FFFFFFFull, "%s: %u x %u outputs", op, a.M, a.N);
    if (grid == 0) return LH_OK;
    constexpr size_t lds = (BN == 256 ? 2 : BM == 256 ? 3 : 5) * (BM + BN) * 128;
    int r = LH_OK;
    with_epilogue(epilogue_of(a.seg, 16), [&](auto epi) {
        constexpr int EPI = decltype(epi)::value;
        const auto kernel = a.ex.tiles ? linear_phased_kernel<BM, BN, EPI, true> : linear_phased_kernel<BM, BN, EPI, false>;
        r = lh_raise_dynamic_lds(ctx, (const void*)kernel, lds, op);
        if (r == LH_OK) hipLaunchKernelGGL(kernel, dim3((uint32_t)grid), dim3(512), lds, ctx->stream, a);
    });
    return r == LH_OK ? lh_check_launch(op) : r;
}

// The forms for the tiles of an expert plan, and what one is expected to take in microseconds: `start`, `step` for each 64 columns of k and, for
// every further tile a CU has, `round` and `round_step`; in each round `through` where a lane cannot store its `lanes` columns as they are, and
// `wide` for f32 results; `empty` for each round of tiles without rows, and `weights` for each 4 MB of them.  Fitted to 1004 products (up to
// 4096 rows, 8192 columns and 128 experts; of 416 the weights came from memory, of the others from the memory-side cache) and then weighed against each
// other: the choice takes 1 % longer than the best form would, on weights from memory 3 %.  64 x 64 tiles come with rings of
// four buffers (up to two workgroups a CU) and of three (three a CU).  Two of 16 experts a row, 2048 -> 1024 columns: 200 rows 18 us (64 x 64; 64 x 32
// tiles that share out k 23), 4096 rows 45 (256 x 256; 128 x 128 of four waves 60).
struct PlanForm {
    uint32_t bm, bn, lanes;
    bool phased;
    float start, step, round, round_step, through, wide, empty, weights;
    int (*launch)(lh_context*, const LhLinear&, uint64_t, const char*);
};
static const PlanForm kPlanForms[] = {
    {256, 256, 16, true, 10.8f, 0.99f, 7.15f, 1.35f, 0.0f, 9.65f, 14.2f, 0.151f, launch_phased<256, 256>},
    {256, 128, 16, true, 11.2f, 0.487f, 6.64f, 0.692f, 0.0f, 8.2f, 0.046f, 0.201f, launch_phased<256, 128>},
    {128, 128, 16, true, 5.99f, 0.545f, 2.7f, 0.567f, 0.0f, 4.1f, 9.55f, 0.0f, launch_phased<128, 128>},
    {128, 128, 16, false, 4.94f, 0.684f, 0.937f, 0.324f, 9.8f, 4.06f, 8.02f, 0.0947f, launch_mfma<128, 128, 2>},
    {64, 64, 8, false, 4.14f, 0.33f, 0.795f, 0.239f, 0.178f, 0.916f, 2.1f, 0.123f, launch_mfma<64, 64, 4>},
    {64, 64, 8, false, 4.04f, 0.366f, 0.49f, 0.204f, 0.0f, 0.984f, 1.71f, 0.115f, launch_mfma<64, 64, 3>},
    {32, 32, 4, false, 5.15f, 0.0526f, 1.41f, 0.102f, 0.0f, 0.35f, 0.611f, 0.577f, launch_sliced<32, 32, 2>},
    {32, 32, 4, false, 4.12f, 0.22f, 0.438f, 0.13f, 0.0f, 0.477f, 0.544f, 0.434f, launch_mfma<32, 32, 4>},
};
static float plan_time(const PlanForm& f, const LhLinear& a, uint64_t steps, uint64_t tiles, uint64_t cus) {
    // A plan has one tile more for each expert than can be full.  Every expert that is chosen has one with rows, and of the last ones about half.
    const uint64_t used = std::min(a.ex.slots, a.ex.experts);
    const uint64_t filled = std::max<uint64_t>(used, a.ex.slots / f.bm + a.ex.experts / 2) * ((a.N + f.bn - 1) / f.bn);
    // Tiles without rows lie between them, so that a CU has one more than its share now and then: a tenth more of the large ones.
    const uint64_t spread = f.bm >= 128 ? filled * 11 / 10 : filled;
    const float rounds = (float)((spread + cus - 1) / cus), s = (float)steps, mb = (float)used * (float)a.N * (float)a.K * 2e-6f;
    return f.start + f.step * s + (rounds - 1) * (f.round + f.round_step * s) +
           rounds * ((epilogue_of(a.seg, f.lanes) == kThroughLds ? f.through : 0.0f) + (a.seg.f32[0] ? f.wide : 0.0f)) +
           (tiles > filled ? f.empty * (float)(tiles - filled) / (float)cus : 0.0f) + f.weights * mb / 4;
}

int lh_launch_linear(lh_context* ctx, const LhLinear& given, const char* op) {
    LhLinear a = given;
    if (a.lda == 0) a.lda = a.K;
    a.parts = 1; a.part_stride = 0;
    const uint32_t a_rows = a.ex.tiles ? (a.ex.gather ? a.ex.rows : a.ex.slots) : a.M, stride = (a.K + 63) / 64 * 64;
    if (a.a_f32 && a.K % 8 == 0 && a.lda % 4 == 0 && (((uintptr_t)a.A | (uintptr_t)a.W) & 15) == 0 && (uint64_t)a_rows * stride * 6 <= ctx->workspace_bytes &&
        a_rows <= 4 * 65535u) {
        if (a_rows == 0) return LH_OK;
        hipLaunchKernelGGL(split_rows_kernel, dim3(split_grid(a_rows, stride, (uint64_t)ctx->cu_count), (a_rows + 3) / 4), dim3(256), 0, ctx->stream, static_cast<const float*>(a.A),
                           static_cast<uint16_t*>(ctx->workspace), a_rows, a.K, a.lda, stride);
        const int r = lh_check_launch(op);
        if (r != LH_OK) return r;
        a.A = ctx->workspace; a.a_f32 = 0; a.lda = 3 * stride; a.parts = 3; a.part_stride = stride;
    }
    const bool mfma = !a.a_f32 && a.K % 8 == 0 && a.lda % 8 == 0 && (((uintptr_t)a.A | (uintptr_t)a.W) & 15) == 0;
    if (!mfma) {
        // (a workgroup for every 64 rows of an expert's tile: 1030 -> 512 columns, 1024 rows with two of 8 experts, 128 rows a workgroup 325 us, 256 637, now 180)
        const uint64_t mt = a.ex.tiles ? (uint64_t)a.ex.n_tiles * (a.ex.tile_rows / 64) : ((uint64_t)a.M + 63) / 64, grid = mt * ((a.N + 63) / 64);
        LH_REQUIRE(grid < 0x7FFFFFFFull, "%s: %u x %u outputs", op, a.M, a.N);
        if (grid == 0) return LH_OK;
        if (a.a_f32) hipLaunchKernelGGL((linear_plain_kernel<float>), dim3((uint32_t)grid), dim3(256), 0, ctx->stream, a);
        else hipLaunchKernelGGL((linear_plain_kernel<uint16_t>), dim3((uint32_t)grid), dim3(256), 0, ctx->stream, a);
        return lh_check_launch(op);
    }
    const uint64_t want = (uint64_t)ctx->cu_count, steps = ((uint64_t)a.K + 63) / 64 * a.parts;
    auto tiles = [&](uint32_t bm, uint32_t bn) {
        return (a.ex.tiles ? (uint64_t)a.ex.n_tiles * (a.ex.tile_rows / bm) : ((uint64_t)a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn);
    };
    // Byte offsets of the phased kernels are 32 bits wide.
    const uint64_t a_bytes = (uint64_t)a_rows * a.lda * 2, w_bytes = (uint64_t)a.N * a.K * 2;
    const bool phased = a.K % 64 == 0 && a_bytes < (1ull << 32) && w_bytes < (1ull << 32);
    if (a.ex.tiles) {
        const PlanForm* best = nullptr;
        float least = INFINITY;
        for (const PlanForm& f : kPlanForms) {
            if ((f.phased && !phased) || a.ex.tile_rows < f.bm) continue;
            const float t = plan_time(f, a, steps, tiles(f.bm, f.bn), want);
            if (t < least) { least = t; best = &f; }
        }
        return best->launch(ctx, a, tiles(best->bm, best->bn), op);
    }
    if (phased && 4 * tiles(128, 128) >= 3 * want) {
        // One workgroup fits a CU, so a launch takes whole rounds of them, and the form is the one whose rounds are the shortest.  A
        // round's time in nanoseconds, measured with 64 columns of k per step: 256 x 256 9000 + 1650 per step, 256 x 128 8000 + 800,
        // 128 x 128 7000 + 520.  Before / now, bf16 results: 2048 x 2048 x 8192 85 / 60 us (256 x 256; the matrix cores alone would take
        // 28 at 2.4 GHz; on random data the clock is 1.5 to 1.8 GHz and they are busy for 70 % of the cycles of such launches), 2048 x 2048 x 4096 39 / 34 and 2048 x 2048 x 3072 35 / 28
        // (256 x 128), 2048 x 8192 x 2048 90 / 74 (128 x 128).  With fewer than three tiles of 128 x 128 to four CUs the small tiles
        // win: 128 of them (953 x 2048 x 2048) 22 us against 18.
        auto rounds = [&](uint32_t bm, uint32_t bn) { return (tiles(bm, bn) + want - 1) / want; };
        const uint64_t t256 = rounds(256, 256) * (9000 + 1650 * steps), t384 = rounds(256, 128) * (8000 + 800 * steps), t128 = rounds(128, 128) * (7000 + 520 * steps);
        if (t256 <= t384 && t256 <= t128) return launch_phased<256, 256>(ctx, a, tiles(256, 256), op);
        if (t384 <= t128) return launch_phased<256, 128>(ctx, a, tiles(256, 128), op);
        return launch_phased<128, 128>(ctx, a, tiles(128, 128), op);
    }
    if (tiles(128, 128) >= 2 * want) return launch_mfma<128, 128, 2>(ctx, a, tiles(128, 128), op);
    // The rest by its expected time in nanoseconds, measured: 64 x 64 or 32 x 32 tiles of shared waves, up to three or five workgroups a CU;
    // waves that share out k, on 64 x 32 tiles (one workgroup a CU) or 32 x 32 (two); or 128 x 64 and 128 x 128 tiles of shared waves, where there is more than
    // one a CU (1702 x 1880 x 2928 41 us on 128 x 64 tiles, weights from memory, 56 on 64 x 64).  A lane that cannot store its columns as they are (bf16 rows that are no multiple of 16 bytes) costs the more the larger the tile.  Before / now,
    // weights in the memory-side cache: 512 x 1024 x 4096 25.5 / 12.5 us, 200 x 2048 x 8192 46.7 / 19.2 and 512 x 1024 x 1024 9.6 / 6.5 (64 x 32), 2048 x 16 x 2048 14.0 / 6.0
    // and 256 x 1024 x 4096 25.2 / 9.4 (32 x 32, shared-out k), 953 x 2048 x 2048 21 / 17.9 and 300 x 6144 x 1536 19.5 / 15.3 (64 x 64, from 128 x 64), 333 x 1024 x 1024
    // with f32 activations 20.3 / 9.6; short k: 287 x 1444 x 176 7.5 / 5.1, 25 x 620 x 136 5.2 / 4.7 (32 x 32, shared waves); ragged k: 3893 x 1504 x 4568 120 / 82 (128 x 128).
    const uint64_t n64 = tiles(64, 64), n32 = tiles(32, 32), n128 = tiles(128, 128), n128_64 = tiles(128, 64);
    auto through = [&](uint32_t lanes, uint64_t t) { return epilogue_of(a.seg, lanes) == kThroughLds ? t : 0; };
    auto per_cu = [&](uint64_t n) { return (n + want - 1) / want; };
    const uint64_t t64 = (n64 <= want ? 4000 + 345 * steps : n64 <= 2 * want ? 4600 + 430 * steps : n64 <= 3 * want ? 5600 + 590 * steps : per_cu(n64) * (2100 + 190 * steps)) + through(8, 1700);
    const uint64_t n6432 = tiles(64, 32), t64_32 = (n6432 <= want ? 4500 + 100 * steps : per_cu(n6432) * (3550 + 148 * steps)) + through(4, 900);
    const uint64_t t32 = (n32 <= want ? 4000 + 75 * steps : 1000 + (n32 + 2 * want - 1) / (2 * want) * (3500 + 150 * steps)) + through(4, 700);
    // (with longer k it is the slower one on weights that come from memory: 200 x 4360 x 1024 18 us against 12 of 64 x 64)
    const uint64_t t32_shared = steps > 4 ? UINT64_MAX : (n32 <= want ? 3700 + 240 * steps : n32 <= 2 * want ? 3900 + 280 * steps : n32 <= 3 * want ? 4300 + 360 * steps : per_cu(n32) * (1100 + 92 * steps)) + through(4, 200);
    const uint64_t t128 = n128 > want ? 8000 + 870 * steps + through(16, 11000) : UINT64_MAX;
    const uint64_t t128_64 = n128_64 > want ? 5800 + 385 * steps + (per_cu(n128_64) - 1) * (1400 + 386 * steps) + through(8, 1700) : UINT64_MAX;
    const uint64_t least = std::min({t64, t64_32, t32, t32_shared, t128_64, t128});
    if (t128_64 == least) return launch_mfma<128, 64, 3>(ctx, a, n128_64, op);
    if (t128 == least) return launch_mfma<128, 128, 2>(ctx, a, n128, op);
    // (with a CU to itself a workgroup keeps four buffers in flight rather than three: 3 % faster, on weights from memory 6 %; from the third a CU on they do not fit, 18 to 30 % slower)
    if (t64 == least) return n64 <= want ? launch_mfma<64, 64, 4>(ctx, a, n64, op) : launch_mfma<64, 64, 3>(ctx, a, n64, op);
    if (t64_32 == least) return launch_sliced<64, 32, 3>(ctx, a, tiles(64, 32), op);
    return t32 == least ? launch_sliced<32, 32, 2>(ctx, a, n32, op) : launch_mfma<32, 32, 4>(ctx, a, n32, op);
}

extern "C" {

int lh_linear_rows_into(lh_batch* batch, const lh_buffer* input, int input_dtype, const lh_buffer* weight, const lh_buffer* bias, uint32_t m, uint32_t k,
                        uint32_t count, const uint32_t* ns, const uint32_t* acts, const uint32_t* heads, const uint32_t* padded, const uint32_t* layouts,
                        lh_buffer* const* outputs, int output_dtype, int accumulate, const lh_buffer* position) {
    const char* op = "linear_rows";
    LH_REQUIRE(batch, "%s: batch is null", op);
    LH_REQUIRE(input_dtype == LH_F32 || input_dtype == LH_BF16, "%s: input dtype %d", op, input_dtype);
    if (m == 0) return LH_OK;
    LhLinear a;
    memset(&a, 0, sizeof a);
    LH_TRY(lh_make_segments(a.seg, op, m, 0, count, ns, acts, heads, padded, layouts, outputs, output_dtype, accumulate, position));
    a.N = a.seg.n0[a.seg.count];
    LH_TRY(check_common(batch, weight, bias, k, a.N, op));
    LH_NEED(input, (size_t)m * k * (input_dtype == LH_F32 ? 4 : 2), op, "input");
    a.A = input->ptr; a.a_f32 = input_dtype == LH_F32;
    a.W = (const uint16_t*)weight->ptr; a.bias = bias ? (const float*)bias->ptr : nullptr;
    a.M = m; a.K = k;
    const int r = lh_launch_linear(batch->ctx, a, op);
    if (r == LH_OK) batch->dispatch_count++;
    return r;
}

int lh_linear_vector_into(lh_batch* batch, const lh_buffer* input, int input_dtype, const lh_buffer* weight, const lh_buffer* bias, uint32_t k,
                          uint32_t count, const uint32_t* ns, const uint32_t* acts, const uint32_t* heads, const uint32_t* padded,
                          const uint32_t* layouts, lh_buffer* const* outputs, int output_dtype, int accumulate, const lh_buffer* position) {
    const char* op = "linear_vector";
    LH_REQUIRE(batch, "%s: batch is null", op);
    LH_REQUIRE(input_dtype == LH_F32 || input_dtype == LH_BF16, "%s: input dtype %d", op, input_dtype);
    LH_NEED(input, (size_t)k * (input_dtype == LH_F32 ? 4 : 2), op, "input");
    VectorStage st{};
    st.x = input->ptr; st.x_f32 = input_dtype == LH_F32;
    return vector_entry(batch, op, kPlain, st, weight, bias, k, count, ns, acts, heads, padded, layouts, outputs, output_dtype, accumulate, position);
}

static int norm_vector(lh_batch* batch, const char* op, const lh_buffer* input, const lh_buffer* add, lh_buffer* store, const lh_buffer* norm_weight, float eps,
                       const lh_buffer* weight, const lh_buffer* bias, uint32_t k, uint32_t count, const uint32_t* ns, const uint32_t* acts,
                       const uint32_t* heads, const uint32_t* padded, const uint32_t* layouts, lh_buffer* const* outputs, int output_dtype,
                       int accumulate, const lh_buffer* position, float cap, lh_buffer* copy = nullptr) {
    LH_REQUIRE(batch, "%s: batch is null", op);
    LH_NEED(input, (size_t)k * 4, op, "input");
    LH_NEED(norm_weight, (size_t)k * 4, op, "norm_weight");
    if (add) LH_NEED(add, (size_t)k * 4, op, "add");
    if (store) {
        LH_NEED(store, (size_t)k * 4, op, "store");
        LH_REQUIRE(store->ptr != input->ptr && (!add || store->ptr != add->ptr), "%s: store must not be read by the other workgroups", op);
    }
    VectorStage st{};
    st.x = input->ptr; st.x_f32 = 1; st.add = add ? (const float*)add->ptr : nullptr; st.store = store ? (float*)store->ptr : nullptr;
    st.norm_weight = (const float*)norm_weight->ptr; st.eps = eps;
    return vector_entry(batch, op, kNorm, st, weight, bias, k, count, ns, acts, heads, padded, layouts, outputs, output_dtype, accumulate, position, cap, copy);
}

int lh_linear_norm_vector_into(lh_batch* batch, const lh_buffer* input, const lh_buffer* add, lh_buffer* store, const lh_buffer* norm_weight, float eps,
                               const lh_buffer* weight, const lh_buffer* bias, uint32_t k, uint32_t count, const uint32_t* ns, const uint32_t* acts,
                               const uint32_t* heads, const uint32_t* padded, const uint32_t* layouts, lh_buffer* const* outputs, int output_dtype,
                               int accumulate, const lh_buffer* position) {
    return norm_vector(batch, "linear_norm_vector", input, add, store, norm_weight, eps, weight, bias, k, count, ns, acts, heads, padded, layouts, outputs, output_dtype,
                       accumulate, position, 0.0f);
}

int lh_linear_norm_vector_capped_into(lh_batch* batch, const lh_buffer* input, const lh_buffer* norm_weight, float eps, const lh_buffer* weight,
                                      const lh_buffer* bias, uint32_t k, uint32_t n, lh_buffer* output, float cap) {
    const char* op = "linear_norm_vector_capped";
    LH_REQUIRE(cap > 0.0f, "%s: cap %g", op, (double)cap);
    const uint32_t act = LH_ACT_NONE, layout = LH_ROWS;
    return norm_vector(batch, op, input, nullptr, nullptr, norm_weight, eps, weight, bias, k, 1, &n, &act, &n, &n, &layout, &output, LH_F32, 0, nullptr, cap);
}

int lh_linear_norm_vector_copied_into(lh_batch* batch, const lh_buffer* input, const lh_buffer* norm_weight, float eps, const lh_buffer* weight,
                                      const lh_buffer* bias, uint32_t k, uint32_t n, lh_buffer* output, lh_buffer* copy, float cap) {
    const char* op = "linear_norm_vector_copied";
    LH_REQUIRE(cap >= 0.0f, "%s: cap %g", op, (double)cap);
    LH_NEED(output, (size_t)n * 4, op, "output");
    LH_NEED(copy, (size_t)n * 4, op, "copy");
    const uint32_t act = LH_ACT_NONE, layout = LH_ROWS;
    return norm_vector(batch, op, input, nullptr, nullptr, norm_weight, eps, weight, bias, k, 1, &n, &act, &n, &n, &layout, &output, LH_F32, 0, nullptr, cap, copy);
}

int lh_linear_residual_norm_vector_copied_into(lh_batch* batch, lh_buffer* input, const lh_buffer* branch, const lh_buffer* branch_weight, float branch_eps,
                                               const lh_buffer* norm_weight, float eps, const lh_buffer* weight, const lh_buffer* bias, uint32_t k, uint32_t n,
                                               lh_buffer* output, lh_buffer* copy, float cap) {
    const char* op = "linear_residual_norm_vector_copied";
    LH_REQUIRE(batch, "%s: batch is null", op);
    LH_REQUIRE(cap >= 0.0f, "%s: cap %g", op, (double)cap);
    LH_NEED(input, (size_t)k * 4, op, "input");
    LH_NEED(branch, (size_t)k * 4, op, "branch");
    LH_NEED(branch_weight, (size_t)k * 4, op, "branch_weight");
    LH_NEED(norm_weight, (size_t)k * 4, op, "norm_weight");
    LH_NEED(output, (size_t)n * 4, op, "output");
    LH_NEED(copy, (size_t)n * 4, op, "copy");
    VectorStage st{};
    st.x = input->ptr; st.x_f32 = 1; st.add = (const float*)branch->ptr; st.norm_weight = (const float*)branch_weight->ptr; st.eps = branch_eps;
    st.outer_weight = (const float*)norm_weight->ptr; st.outer_eps = eps;
    const uint64_t cus = (uint64_t)batch->ctx->cu_count;
    if (k % 8 == 0 && k > 0 && copied_in_product(k, n) && n > 8 * cus && weight && ((uintptr_t)weight->ptr & 15) == 0 && lh_stage_aligned(st)) {
        LH_TRY(check_common(batch, weight, bias, k, n, op));
        LhSegments seg;
        const uint32_t act = LH_ACT_NONE, layout = LH_ROWS;
        LH_TRY(lh_make_segments(seg, op, 1, 0, 1, &n, &act, &n, &n, &layout, &output, LH_F32, 0, nullptr));
        seg.cap = cap;
        const uint32_t grid = one_row_grid(n, k, 8, 64, cus);
#define LH_MVC(NLOADS) hipLaunchKernelGGL((matvec_bf16_reg_kernel<kResidualNorm, NLOADS, 8, true>), dim3(grid), dim3(512), 0, batch->ctx->stream, st, (const uint16_t*)weight->ptr, \
                                          bias ? (const float*)bias->ptr : nullptr, seg, n, k, (float*)copy->ptr)
        if (k <= 512) LH_MVC(1);
        else if (k <= 1024) LH_MVC(2);
        else LH_MVC(4);
#undef LH_MVC
        const int r = lh_check_launch(op);
        if (r == LH_OK) batch->dispatch_count++;
        return r;
    }
    LH_TRY(lh_residual_rows_into(batch, input, branch, branch_weight, input, nullptr, LH_F32, k, 1, branch_eps));
    return lh_linear_norm_vector_copied_into(batch, input, norm_weight, eps, weight, bias, k, n, output, copy, cap);
}

int lh_linear_residual_vector_into(lh_batch* batch, const lh_buffer* input, const lh_buffer* branch, lh_buffer* store, const lh_buffer* norm_weight,
                                   float eps, const lh_buffer* weight, const lh_buffer* bias, uint32_t k, uint32_t count, const uint32_t* ns,
                                   const uint32_t* acts, const uint32_t* heads, const uint32_t* padded, const uint32_t* layouts, lh_buffer* const* outputs,
                                   int output_dtype, int accumulate, const lh_buffer* position) {
    const char* op = "linear_residual_vector";
    LH_REQUIRE(batch, "%s: batch is null", op);
    LH_NEED(input, (size_t)k * 4, op, "input");
    LH_NEED(branch, (size_t)k * 4, op, "branch");
    LH_NEED(norm_weight, (size_t)k * 4, op, "norm_weight");
    if (store) {
        LH_NEED(store, (size_t)k * 4, op, "store");
        LH_REQUIRE(store->ptr != input->ptr && store->ptr != branch->ptr, "%s: store must not be read by the other workgroups", op);
    }
    VectorStage st{};
    st.x = input->ptr; st.x_f32 = 1; st.add = (const float*)branch->ptr; st.store = store ? (float*)store->ptr : nullptr;
    st.norm_weight = (const float*)norm_weight->ptr; st.eps = eps;
    return vector_entry(batch, op, kResidual, st, weight, bias, k, count, ns, acts, heads, padded, layouts, outputs, output_dtype, accumulate, position);
}

uint32_t lh_gated_vector_fits(uint32_t k, uint32_t group) {
    if (group == k) return 1;
    if (group == 0 || k % group || group % 8 || k > 4096) return 0;
    const uint32_t c = group / 8;
    return c % 64 == 0 || (c < 64 && (c & (c - 1)) == 0);
}

int lh_linear_gated_vector_into(lh_batch* batch, const lh_buffer* input, const lh_buffer* gate, int gate_dtype, uint32_t gate_act, int gate_first,
                                const lh_buffer* norm_weight, uint32_t group, float eps, const lh_buffer* weight, const lh_buffer* bias, uint32_t k, uint32_t count, const uint32_t* ns, const uint32_t* acts,
                                const uint32_t* heads, const uint32_t* padded, const uint32_t* layouts, lh_buffer* const* outputs, int output_dtype,
                                int accumulate, const lh_buffer* position) {
    const char* op = "linear_gated_vector";
    LH_REQUIRE(batch, "%s: batch is null", op);
    LH_REQUIRE(gate_dtype == LH_F32 || gate_dtype == LH_BF16, "%s: gate dtype %d", op, gate_dtype);
    LH_NEED(input, (size_t)k * 4, op, "input");
    LH_NEED(gate, (size_t)k * (gate_dtype == LH_F32 ? 4 : 2), op, "gate");
    if (norm_weight) LH_NEED(norm_weight, (size_t)k * 4, op, "norm_weight");
    LH_REQUIRE(gate_act == LH_ACT_SIGMOID || gate_act == LH_ACT_SILU, "%s: gate activation %u", op, gate_act);
    LH_REQUIRE(lh_gated_vector_fits(k, group), "%s: %u values in parts of %u", op, k, group);
    VectorStage st{};
    st.x = input->ptr; st.x_f32 = 1; st.norm_weight = norm_weight ? (const float*)norm_weight->ptr : nullptr; st.gate = gate->ptr;
    st.gate_f32 = gate_dtype == LH_F32; st.gate_act = gate_act; st.gate_first = gate_first != 0; st.group = group; st.eps = eps;
    LH_REQUIRE(group == k || lh_stage_aligned(st), "%s: buffers must be 16-byte aligned", op);
    LH_REQUIRE(group == k || ((uintptr_t)weight->ptr & 15) == 0, "%s: the weight must be 16-byte aligned", op);
    return vector_entry(batch, op, kGated, st, weight, bias, k, count, ns, acts, heads, padded, layouts, outputs, output_dtype, accumulate, position);
}

}  // extern "C"
