// Internal interface of the bf16-weight products (float_linear.hip) for the mixture-of-experts entries (float_moe.hip).
#pragma once
#include "float_ops.hpp"

// Rows of an expert product: the plan's tiles (see float_moe.hip), each `tile_rows` plan slots of one expert.
struct LhExpertRows {
    const uint32_t* tiles;          // null: an ordinary product.  [n_tiles][3]: expert, first slot, one past the last slot
    uint32_t n_tiles, tile_rows;    // 64, 128 or 256
    const uint32_t* slot_row;       // slot -> row of the activations
    const float* slot_weight;       // slot -> weight of the expert's input (null: 1)
    uint32_t gather;                // activations are indexed by slot_row (else by the slot itself)
    uint32_t scatter;               // outputs go to slot_row (else to the slot itself)
    uint32_t experts, slots, rows;  // bounds of the above
};

struct LhLinear {
    const void* A;                  // [M, K], bf16 or f32, rows `lda` elements apart (0: K)
    uint32_t a_f32;
    const uint16_t* W;              // [N, K] (of every expert, one after the other)
    const float* bias;
    uint32_t M, N, K, lda;
    uint32_t parts, part_stride;    // bf16 rows that hold K columns `parts` times (0: once), part_stride elements apart: terms of f32 values
    LhSegments seg;
    LhExpertRows ex;
};
int lh_launch_linear(lh_context* ctx, const LhLinear& a, const char* op);
uint32_t lh_expert_tile_rows(uint32_t slots, uint32_t experts);

// ---- one row: the activation vector in registers -------------------------------------------------------------------------
// Up to 4096 columns a wave keeps the vector itself: lane l holds the NL chunks of eight elements 8 (64 c + l), which is what
// it multiplies in every row.
enum { kPlain = 0, kNorm = 1, kGated = 2, kResidual = 3, kResidualNorm = 4 };   // the last: a residual, and the norm of it
struct VectorStage {
    const void* x;             // plain: x_f32 ? f32 : bf16; the others: f32
    uint32_t x_f32;
    const float* add;          // norm: may be null; residual: what is normed and added
    float* store;              // norm, residual: receives the sum (workgroup 0), may be null
    const float* norm_weight;  // gated: may be null
    union {
        const void* gate;            // gated
        const float* outer_weight;   // residual and norm: of the norm
    };
    uint32_t gate_f32, gate_act, gate_first;          // gated: the gate multiplies before the norm
    union {
        uint32_t group;              // gated: elements per normed part
        float outer_eps;             // residual and norm
    };
    float eps;
};

__device__ __forceinline__ void lh_ld8(const float* p, float (&v)[8]) {
    const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ void lh_ld8(const uint16_t* p, float (&v)[8]) {
    const uint4 a = *reinterpret_cast<const uint4*>(p);
    const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
    for (int j = 0; j < 4; j++) { v[2 * j] = __builtin_bit_cast(float, w[j] << 16); v[2 * j + 1] = __builtin_bit_cast(float, w[j] & 0xFFFF0000u); }
}

// A vector for the registers of W waves, K a multiple of 8 up to 512 NL, all pointers 16-byte aligned, zero past K: wave c brings in
// the chunks 64 c + lane and what they need, the sums of the norm meet in LDS, and every wave takes the finished vector from there.
// (Every wave for itself: 16 KB from the caches per wave for 2048 columns with a norm, as much as the weights of two rows.)  Up to 512
// columns, a chunk a lane, every wave does bring it in for itself: there the barriers are what takes the time (512 x 512 behind a
// norm with eight waves: 3.3 us with them, 3.1 without).
//
// Loads return in order, so what is requested first can be waited for alone: the vector first (`fetch`), then the weights of the first
// rows, then `finish`.  And behind a load that not every path makes the compiler waits for all there are, so every load here is
// made: lanes and waves without a chunk load one that exists, and an operand that is not there is read from x.
constexpr int kVectorWaves = 8;
template <int W = kVectorWaves> struct LhVectorSpace { float4 x[2 * W][64]; float part[W], outer[W]; };

// Eight values at element k, stored as f32 or bf16.
struct LhEither8 {
    uint4 a, b;
    __device__ __forceinline__ void load(const void* p, bool f32, uint32_t k) {
        const char* q = static_cast<const char*>(p) + (size_t)k * (f32 ? 4 : 2);
        a = *reinterpret_cast<const uint4*>(q);
        b = *reinterpret_cast<const uint4*>(q + (f32 ? 16 : 0));
    }
    __device__ __forceinline__ void get(bool f32, float (&v)[8]) const {
        const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = __builtin_bit_cast(float, f32 ? w[j] : j & 1 ? w[j >> 1] & 0xFFFF0000u : w[j >> 1] << 16);
    }
};

template <int STAGE, int NL, int W = kVectorWaves>
struct LhSharedVector {
    static_assert(NL <= W, "a chunk per wave");
    static constexpr bool kAlone = NL == 1;
    static constexpr bool kAround = STAGE == kResidualNorm, kBranch = STAGE == kResidual || kAround;
    static constexpr bool kNormed = STAGE == kNorm || STAGE == kGated || kBranch;
    static constexpr bool kAdds = STAGE == kNorm || kBranch;
    LhEither8 x, gate;
    float w[8], more[8], around[8];

    __device__ __forceinline__ void fetch(const VectorStage& st, uint32_t K, uint32_t lane, uint32_t wave) {
        const uint32_t k = kAlone ? min(lane * 8, K - 8) : wave < NL ? min((64 * wave + lane) * 8, K - 8) : 0u;
        x.load(st.x, STAGE != kPlain || st.x_f32, k);
        if constexpr (kNormed) lh_ld8((st.norm_weight ? st.norm_weight : static_cast<const float*>(st.x)) + k, w);
        if constexpr (kAdds) lh_ld8((st.add ? st.add : static_cast<const float*>(st.x)) + k, more);
        if constexpr (STAGE == kGated) gate.load(st.gate, st.gate_f32, k);
        if constexpr (kAround) lh_ld8(st.outer_weight + k, around);
    }
    __device__ __forceinline__ void finish(const VectorStage& st, uint32_t K, uint32_t lane, uint32_t wave, bool store, LhVectorSpace<W>& sp, float (&xr)[NL][8]) {
        const uint32_t k = (64 * (kAlone ? 0u : wave) + lane) * 8;
        const bool owner = kAlone || wave < NL, in = owner && k < K;
        float v[8], sum = 0.0f;
        x.get(STAGE != kPlain || st.x_f32, v);
        if constexpr (STAGE == kNorm)
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = st.add ? v[j] + more[j] : v[j];
        if constexpr (STAGE == kGated) {
            float g[8];
            gate.get(st.gate_f32, g);
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const float f = lh_gate(g[j], st.gate_act);
                w[j] = st.norm_weight ? w[j] : 1.0f;
                if (st.gate_first) v[j] *= f; else w[j] *= f;
            }
        }
        if constexpr (kNormed) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                if constexpr (kBranch) { sum += more[j] * more[j]; w[j] *= more[j]; }      // the weighted branch
                else sum += v[j] * v[j];
            }
            sum = in ? sum : 0.0f;
            const bool parts = STAGE == kGated && st.group != K;   // group / 8 chunks: a power of two of lanes, or whole sets of 64
            const uint32_t cg = parts ? st.group >> 3 : 64u, width = min(cg, 64u);
            sum = lh_group_sum(sum, (int)width);
            if (!kAlone && width == 64) {
                if (lane == 0) sp.part[wave] = sum;
                lh_lds_barrier();
                const uint32_t per = parts ? cg >> 6 : (uint32_t)W, w0 = wave / per;
                sum = 0.0f;
#pragma unroll
                for (int e = 0; e < W; e++) sum += (uint32_t)e / per == w0 ? sp.part[e] : 0.0f;
            }
            const float r = rsqrtf(sum / (float)(parts ? st.group : K) + st.eps);
            if constexpr (kBranch)
#pragma unroll
                for (int j = 0; j < 8; j++) v[j] = __builtin_fmaf(w[j], r, v[j]);
            if (STAGE != kGated && store && in && (!kAlone || wave == 0)) {
                *reinterpret_cast<float4*>(st.store + k) = make_float4(v[0], v[1], v[2], v[3]);
                *reinterpret_cast<float4*>(st.store + k + 4) = make_float4(v[4], v[5], v[6], v[7]);
            }
            if constexpr (!kBranch)
#pragma unroll
                for (int j = 0; j < 8; j++) v[j] = v[j] * r * w[j];
            if constexpr (kAround) {
                float s = 0.0f;
#pragma unroll
                for (int j = 0; j < 8; j++) s += v[j] * v[j];
                s = lh_group_sum(in ? s : 0.0f, 64);
                if constexpr (!kAlone) {
                    if (lane == 0) sp.outer[wave] = s;
                    lh_lds_barrier();
                    s = 0.0f;
#pragma unroll
                    for (int e = 0; e < W; e++) s += sp.outer[e];
                }
                const float f = rsqrtf(s / (float)K + st.outer_eps);
#pragma unroll
                for (int j = 0; j < 8; j++) v[j] = v[j] * f * around[j];
            }
        }
        if constexpr (kAlone) {
#pragma unroll
            for (int j = 0; j < 8; j++) xr[0][j] = in ? v[j] : 0.0f;
            return;
        }
        if (owner) {
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = in ? v[j] : 0.0f;
            sp.x[2 * wave][lane] = make_float4(v[0], v[1], v[2], v[3]);
            sp.x[2 * wave + 1][lane] = make_float4(v[4], v[5], v[6], v[7]);
        }
        lh_lds_barrier();
#pragma unroll
        for (int c = 0; c < NL; c++) {
            const float4 a = sp.x[2 * c][lane], b = sp.x[2 * c + 1][lane];
            xr[c][0] = a.x; xr[c][1] = a.y; xr[c][2] = a.z; xr[c][3] = a.w; xr[c][4] = b.x; xr[c][5] = b.y; xr[c][6] = b.z; xr[c][7] = b.w;
        }
    }
};

static inline bool lh_stage_aligned(const VectorStage& st) {
    return (((uintptr_t)st.x | (uintptr_t)st.add | (uintptr_t)st.store | (uintptr_t)st.norm_weight | (uintptr_t)st.gate) & 15) == 0;
}

// Weights are read once per launch: streaming loads.
__device__ __forceinline__ uint4 lh_ld16_stream(const uint16_t* p) {
    typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
    const u32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ float lh_dot8(const uint4& v, const float* x, float acc) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int j = 0; j < 4; j++) {
        acc = __builtin_fmaf(__builtin_bit_cast(float, w[j] << 16), x[2 * j], acc);
        acc = __builtin_fmaf(__builtin_bit_cast(float, w[j] & 0xFFFF0000u), x[2 * j + 1], acc);
    }
    return acc;
}
