// Linear attention with a decay a per head: for every token M <- a M + k (x) v, y = q M.  The decay is fixed, or computed from
// the token together with a step size that scales k (x) v (selective state space; heads may then share q and k in groups, and
// a multiple of v is added to y).  The state M is f32,
// kept as [head][value column][DQ key columns] (the key columns that exist, then zeros).
//
// Recurrent form: a wave (65 to 512 key columns) or a row of 16 lanes holds one value column's state in registers and walks the
// rows, whose inputs come in several rows ahead.
//
// Chunked form (64 or 128 rows a chunk, bf16 inputs on the matrix cores, everything else f32; with 128 the states, which every step
// writes or reads, are half as many):
//   1. every chunk's own contribution to the state, U = sum over rows s of a^(L-1-s) k_s (x) v_s (all chunks at once)
//   2. a scan over the chunks, M <- a^L M + U, that leaves each chunk's incoming state in place of its U
//   3. all outputs: y_t = a^(t+1) q_t M_in + sum over s <= t of a^(t-s) (q_t . k_s) v_s
// With decays per token, a power becomes the exponential of a difference of running sums of the decays' logarithms.
// Where an f32 quantity enters a product (decayed keys, decayed scores, the state) it does so as the sum of three bf16
// terms, which is all of its 24 bits; the products of bf16 values are exact and summed in f32.
#include "float_ops.hpp"
#include <algorithm>

namespace {

constexpr uint32_t kHalf = 64;   // rows that the callers' powers, and the running sums of a selective state space, reach over: a chunk or half of one

// What the step of a token is: fixed per head, or computed from the token (selective state space).
__device__ __forceinline__ float softplus(float z) { return fmaxf(z, 0.0f) + log1pf(expf(-fabsf(z))); }

// Where the decay comes from is known when a kernel is compiled, so that a token's launch starts with no address to compute from a stride.
enum Decay { kFixed, kPowers, kSelective };

struct RecurrentArgs {
    const void *q, *k, *v;
    float* state;
    const float* decay;                                     // [heads], or [heads, kHalf + 1] powers of them
    const float *dt_raw, *dt_bias, *a_log, *skip;           // selective: [rows, heads], then [heads] each
    float* out;
    uint32_t rows, heads, key_heads, dim, dq, vdim;
    float scale;
};

template <typename T, int NR, Decay DECAY>
__global__ __launch_bounds__(256) void recurrent_kernel(const RecurrentArgs a) {
    constexpr bool SELECTIVE = DECAY == kSelective;
    const T *q = static_cast<const T*>(a.q), *k = static_cast<const T*>(a.k), *v = static_cast<const T*>(a.v);
    const uint32_t dim = a.dim, dq = a.dq, vdim = a.vdim, heads = a.heads, rows = a.rows;
    const uint32_t vt = (vdim + 15) / 16, h = blockIdx.x / vt, col = (blockIdx.x % vt) * 16 + (threadIdx.x >> 4), part = threadIdx.x & 15;
    const uint32_t kh = h / (heads / a.key_heads);
    const bool on = col < vdim;
    const uint32_t c = on ? col : vdim - 1, k0 = part * NR;
    float* st = a.state + ((size_t)h * vdim + c) * dq + k0;
    float s[NR];
#pragma unroll
    for (int i = 0; i < NR; i++) s[i] = k0 + i < dq ? st[i] : 0.0f;
    const float fixed = SELECTIVE ? 0.0f : a.decay[(size_t)h * (DECAY == kPowers ? kHalf + 1 : 1)], rate = SELECTIVE ? -expf(a.a_log[h]) : 0.0f, bias = SELECTIVE ? a.dt_bias[h] : 0.0f,
                skip = SELECTIVE ? a.skip[h] : 0.0f;
    float kn[NR], qn[NR], vn, zn = 0.0f;
    auto fetch = [&](uint32_t t) {
        const size_t row = ((size_t)t * a.key_heads + kh) * dq + k0;
#pragma unroll
        for (int i = 0; i < NR; i++) {
            const bool in = k0 + i < dim;
            kn[i] = in ? lh_ld(k, row + i) : 0.0f;
            qn[i] = in ? lh_ld(q, row + i) : 0.0f;
        }
        vn = lh_ld(v, ((size_t)t * heads + h) * vdim + c);
        if (SELECTIVE) zn = a.dt_raw[(size_t)t * heads + h];
    };
    fetch(0);
    for (uint32_t t = 0; t < rows; t++) {
        float kc[NR], qc[NR];
        const float x = vn, dt = SELECTIVE ? softplus(zn + bias) : 1.0f, d = SELECTIVE ? expf(rate * dt) : fixed, vc = SELECTIVE ? dt * x : x;
#pragma unroll
        for (int i = 0; i < NR; i++) { kc[i] = kn[i]; qc[i] = qn[i]; }
        if (t + 1 < rows) fetch(t + 1);
        float o = 0.0f;
#pragma unroll
        for (int i = 0; i < NR; i++) {
            s[i] = __builtin_fmaf(kc[i], vc, d * s[i]);
            o = __builtin_fmaf(s[i], qc[i], o);
        }
        o = lh_group_sum(o, 16);
        if (part == 0 && on) a.out[((size_t)t * heads + h) * vdim + col] = SELECTIVE ? __builtin_fmaf(skip, x, o) : o * a.scale;
    }
    if (on) {
#pragma unroll
        for (int i = 0; i < NR; i++) if (k0 + i < dq) st[i] = s[i];
    }
}

// N neighbouring values, as they are stored.
template <typename T, int N> struct Packed;
template <int N> struct Packed<float, N> {
    float v[N];
    __device__ __forceinline__ void load(const float* p) {
        if constexpr (N == 2) { const float2 x = *reinterpret_cast<const float2*>(p); v[0] = x.x; v[1] = x.y; }
        else
#pragma unroll
            for (int i = 0; i < N; i += 4) { const float4 x = *reinterpret_cast<const float4*>(p + i); v[i] = x.x; v[i + 1] = x.y; v[i + 2] = x.z; v[i + 3] = x.w; }
    }
    __device__ __forceinline__ float get(int i) const { return v[i]; }
};
template <int N> struct Packed<uint16_t, N> {
    uint32_t v[N / 2];
    __device__ __forceinline__ void load(const uint16_t* p) {
        if constexpr (N == 2) v[0] = *reinterpret_cast<const uint32_t*>(p);
        else if constexpr (N == 4) { const uint2 x = *reinterpret_cast<const uint2*>(p); v[0] = x.x; v[1] = x.y; }
        else
#pragma unroll
            for (int i = 0; i < N / 2; i += 4) { const uint4 x = *reinterpret_cast<const uint4*>(p + 2 * i); v[i] = x.x; v[i + 1] = x.y; v[i + 2] = x.z; v[i + 3] = x.w; }
    }
    __device__ __forceinline__ float get(int i) const { return __builtin_bit_cast(float, i & 1 ? v[i >> 1] & 0xFFFF0000u : v[i >> 1] << 16); }
};

// The same recurrence over many rows.  A step is a few dozen instructions behind its inputs, so the inputs of AHEAD rows are on their
// way at any time, in whole pieces, and no load is conditional (one row ahead and a value at a time: 2 us a row; now 0.2).
template <typename T, int NR, int AHEAD, Decay DECAY>
__global__ __launch_bounds__(256) void recurrent_rows_kernel(const RecurrentArgs a) {
    constexpr bool SELECTIVE = DECAY == kSelective;
    const uint32_t dim = a.dim, dq = a.dq, vdim = a.vdim, heads = a.heads, rows = a.rows;
    const uint32_t vt = (vdim + 15) / 16, h = blockIdx.x / vt, col = (blockIdx.x % vt) * 16 + (threadIdx.x >> 4), part = threadIdx.x & 15;
    const bool on = col < vdim, has = part * NR < dq;             // (dq is a multiple of NR: a lane has all of its values, or none)
    const uint32_t c = on ? col : vdim - 1, k0 = has ? part * NR : 0u, in = !has ? 0u : k0 < dim ? min(dim - k0, (uint32_t)NR) : 0u;
    const size_t step = (size_t)a.key_heads * dq, first = (size_t)(h / (heads / a.key_heads)) * dq + k0;
    const T *q = static_cast<const T*>(a.q) + first, *k = static_cast<const T*>(a.k) + first, *v = static_cast<const T*>(a.v) + (size_t)h * vdim + c;
    float* st = a.state + ((size_t)h * vdim + c) * dq + k0;
    float s[NR];
#pragma unroll
    for (int i = 0; i < NR; i++) s[i] = has ? st[i] : 0.0f;
    const float fixed = SELECTIVE ? 0.0f : a.decay[(size_t)h * (DECAY == kPowers ? kHalf + 1 : 1)], rate = SELECTIVE ? -expf(a.a_log[h]) : 0.0f, bias = SELECTIVE ? a.dt_bias[h] : 0.0f,
                skip = SELECTIVE ? a.skip[h] : 0.0f;
    struct Row { Packed<T, NR> k, q; T v; float z; } next[AHEAD];
    auto fetch = [&](Row& r, uint32_t t) {
        const size_t u = min(t, rows - 1);
        r.k.load(k + u * step);
        r.q.load(q + u * step);
        r.v = v[u * heads * vdim];
        if (SELECTIVE) r.z = a.dt_raw[u * heads + h];
    };
    auto walk = [&](const Row& r, uint32_t t) {
        const float x = lh_ld(&r.v, 0), dt = SELECTIVE ? softplus(r.z + bias) : 1.0f, d = SELECTIVE ? expf(rate * dt) : fixed, vc = SELECTIVE ? dt * x : x;
        float o = 0.0f;
#pragma unroll
        for (int i = 0; i < NR; i++) {
            s[i] = __builtin_fmaf((uint32_t)i < in ? r.k.get(i) : 0.0f, vc, d * s[i]);
            o = __builtin_fmaf(s[i], (uint32_t)i < in ? r.q.get(i) : 0.0f, o);
        }
        o = lh_group_sum(o, 16);
        if (part == 0 && on) a.out[((size_t)t * heads + h) * vdim + col] = SELECTIVE ? __builtin_fmaf(skip, x, o) : o * a.scale;
    };
#pragma unroll
    for (int j = 0; j < AHEAD; j++) fetch(next[j], j);
    uint32_t t = 0;
    for (; t + AHEAD <= rows; t += AHEAD) {
#pragma unroll
        for (int j = 0; j < AHEAD; j++) {
            walk(next[j], t + j);
            fetch(next[j], t + AHEAD + j);
        }
    }
#pragma unroll
    for (int j = 0; j < AHEAD; j++) if (t + j < rows) walk(next[j], t + j);
    if (on && has) {
#pragma unroll
        for (int i = 0; i < NR; i++) st[i] = s[i];
    }
}

// The same with a wave a value column: four times as many waves, a quarter of the state in each.  Where columns are few the form above has a
// wave on every fourth SIMD, and a row is the instructions of one wave one behind the other: 333 rows of 8 heads, 128 x 128, in 32 bits
// 62 us there (450 cycles a row), 31 here.  Four rows' sums over the lanes share their steps -- a lane keeps the row of its two lowest bits --
// and leave in one store; what a selective state space computes for a row is computed for AHEAD rows at a time, a lane each.
template <typename T, int NR, int AHEAD, Decay DECAY>
__global__ __launch_bounds__(256) void recurrent_wide_kernel(const RecurrentArgs a) {
    static_assert(AHEAD % 4 == 0 && AHEAD <= 64, "rows in fours, a lane each");
    constexpr bool SELECTIVE = DECAY == kSelective;
    const uint32_t lane = threadIdx.x & 63, column = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), dim = a.dim, dq = a.dq, vdim = a.vdim, heads = a.heads, rows = a.rows;
    if (column >= heads * vdim) return;
    const uint32_t h = column / vdim;
    const bool has = lane * NR < dq;                              // (dq is a multiple of NR: a lane has all of its values, or none)
    const uint32_t k0 = has ? lane * NR : 0u, in = !has ? 0u : k0 < dim ? min(dim - k0, (uint32_t)NR) : 0u;
    const size_t step = (size_t)a.key_heads * dq, first = (size_t)(h / (heads / a.key_heads)) * dq, across = (size_t)heads * vdim;
    const T *q = static_cast<const T*>(a.q) + first, *k = static_cast<const T*>(a.k) + first, *v = static_cast<const T*>(a.v) + column;
    float* st = a.state + (size_t)column * dq;
    float s[NR];
#pragma unroll
    for (int i = 0; i < NR; i++) s[i] = has ? st[k0 + i] : 0.0f;
    const float fixed = SELECTIVE ? 0.0f : a.decay[(size_t)h * (DECAY == kPowers ? kHalf + 1 : 1)], rate = SELECTIVE ? -expf(a.a_log[h]) : 0.0f, bias = SELECTIVE ? a.dt_bias[h] : 0.0f,
                skip = SELECTIVE ? a.skip[h] : 0.0f;
    struct Row { Packed<T, NR> k, q; T v; } next[AHEAD];
    auto fetch = [&](Row& r, uint32_t t) {
        const size_t u = min(t, rows - 1);
        r.k.load(k + u * step + k0);
        r.q.load(q + u * step + k0);
        r.v = v[u * across];
    };
    auto raw = [&](uint32_t t) { return SELECTIVE ? a.dt_raw[(size_t)min(t + min(lane, (uint32_t)AHEAD - 1), rows - 1) * heads + h] : 0.0f; };
    float z = raw(0), dts = 1.0f, ds = 1.0f;                        // lane j: what row t + j has
    auto steps = [&](uint32_t t) {                                  // of rows t .. t + AHEAD - 1; the next ones' are requested
        if constexpr (SELECTIVE) {
            dts = softplus(z + bias);
            ds = expf(rate * dts);
            z = raw(t + AHEAD);
        }
    };
    auto at_row = [&](float x, int j) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), j)); };
    auto four = [&](const Row* r, int j0, uint32_t t, uint32_t count) {
        float o[4], x[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            o[j] = 0.0f;
            x[j] = lh_ld(&r[j].v, 0);
            if ((uint32_t)j >= count) continue;
            const float dt = SELECTIVE ? at_row(dts, j0 + j) : 1.0f, d = SELECTIVE ? at_row(ds, j0 + j) : fixed, vc = SELECTIVE ? dt * x[j] : x[j];
#pragma unroll
            for (int i = 0; i < NR; i++) {
                s[i] = __builtin_fmaf((uint32_t)i < in ? r[j].k.get(i) : 0.0f, vc, d * s[i]);
                o[j] = __builtin_fmaf(s[i], (uint32_t)i < in ? r[j].q.get(i) : 0.0f, o[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < 4; j++) o[j] += lh_dpp_f<LH_DPP_QUAD_XOR1>(o[j]);
        float e = lane & 1 ? o[1] : o[0], f = lane & 1 ? o[3] : o[2];
        e += lh_dpp_f<LH_DPP_QUAD_XOR2>(e);
        f += lh_dpp_f<LH_DPP_QUAD_XOR2>(f);
        float y = lane & 2 ? f : e;
        y += lh_lane_xor_f<4>(y);
        y += lh_lane_xor_f<8>(y);
        y = lh_sum32_f(lh_sum16_f(y));
        if (SELECTIVE) y = __builtin_fmaf(skip, lane & 2 ? (lane & 1 ? x[3] : x[2]) : (lane & 1 ? x[1] : x[0]), y);
        else y *= a.scale;
        if (lane < count) a.out[(size_t)(t + lane) * across + column] = y;
    };
#pragma unroll
    for (int j = 0; j < AHEAD; j++) fetch(next[j], j);
    uint32_t t = 0;
    for (; t + AHEAD <= rows; t += AHEAD) {
        steps(t);
#pragma unroll
        for (int j = 0; j < AHEAD; j += 4) {
            four(next + j, j, t + j, 4);
#pragma unroll
            for (int i = 0; i < 4; i++) fetch(next[j + i], t + AHEAD + j + i);
        }
    }
    steps(t);
#pragma unroll
    for (int j = 0; j < AHEAD; j += 4) if (t + j < rows) four(next + j, j, t + j, min(rows - t - j, 4u));
    if (has) {
#pragma unroll
        for (int i = 0; i < NR; i++) st[k0 + i] = s[i];
    }
}

// The steps of a selective state space, one wave per head and 64 rows: step sizes, and the running sum of the logarithms of the
// decays within those rows.  Rows past the last have step 0 and decay 1.
__global__ __launch_bounds__(64) void chunk_steps_kernel(const float* __restrict__ dt_raw, const float* __restrict__ dt_bias, const float* __restrict__ a_log,
                                                        float* __restrict__ sums, float* __restrict__ sizes, uint32_t rows, uint32_t heads, uint32_t halves) {
    const uint32_t h = blockIdx.x % heads, c = blockIdx.x / heads, lane = threadIdx.x, t = c * kHalf + lane;
    const float dt = t < rows ? softplus(dt_raw[(size_t)t * heads + h] + dt_bias[h]) : 0.0f;
    float sum = -expf(a_log[h]) * dt;
#pragma unroll
    for (uint32_t d = 1; d < 64; d <<= 1) {
        const float o = __shfl_up(sum, d, 64);
        if (lane >= d) sum += o;
    }
    const size_t i = ((size_t)h * halves + c) * kHalf + lane;
    sums[i] = sum;
    sizes[i] = dt;
}

struct ChunkArgs {
    const uint16_t *q, *k, *v;
    float* state;
    const float* powers;       // fixed decays: [heads][65]
    const float *sums, *sizes; // selective: [heads][halves][64]
    const float* skip;         // selective: [heads]
    float* chunk_state;        // [chunk][heads][vdim][dq]
    float* out;
    uint32_t rows, heads, key_heads, dim, vdim, chunk, chunks, halves;    // `chunk`: rows of one, 64 or 128
    float scale;
};

// A decay from one half of a chunk into the other is taken in two steps, to the end of the first half and on from there: neither power
// is above the callers' 64, so that what is finite in steps of 64 rows stays so with decays above one, and differences of running sums
// keep their bits.

__device__ __forceinline__ lh_bf16x8 bf8(const uint32_t (&w)[4]) {
    struct { uint32_t v[4]; } t = {{w[0], w[1], w[2], w[3]}};
    return __builtin_bit_cast(lh_bf16x8, t);
}
// Two values as three bf16 terms each, the first value's in the lower halves.
__device__ __forceinline__ void split3_pair(float a, float b, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
    hi = lh_pack_bf(a, b);
    const float ra = a - __builtin_bit_cast(float, hi << 16), rb = b - __builtin_bit_cast(float, hi & 0xFFFF0000u);
    mid = lh_pack_bf(ra, rb);
    lo = lh_pack_bf(ra - __builtin_bit_cast(float, mid << 16), rb - __builtin_bit_cast(float, mid & 0xFFFF0000u));
}
// Element j of the rows in a (lower half) and b (upper half).
__device__ __forceinline__ uint32_t pick(const uint2& a, const uint2& b, int j) {
    return __builtin_amdgcn_perm(j & 2 ? b.y : b.x, j & 2 ? a.y : a.x, j & 1 ? 0x07060302u : 0x05040100u);
}

// What lies `offset` bytes behind a base that is the same for the whole wave.
template <typename T> __device__ __forceinline__ T at(const void* base, uint32_t offset) { return *reinterpret_cast<const T*>(static_cast<const char*>(base) + offset); }
// Four neighbouring columns of a row of values from `col`, no further than the last column: where there is none, what comes is not
// used.  (No load below is conditional: a branch around it would wait for it.)  VALUES: kPieces, the columns a multiple of four;
// kWords, any four columns or more, the last four of the row shifted into place (a column at a time: 24.9 us for 2048 rows of 3 heads of
// 20 x 33, all three kernels; now 15.0); kSingles, fewer than four.
enum Values { kPieces, kWords, kSingles };
template <Values VALUES> __device__ __forceinline__ uint2 load_values(const uint16_t* base, uint32_t row_offset, uint32_t col, uint32_t vdim) {
    if constexpr (VALUES == kPieces) return at<uint2>(base, row_offset + 2 * min(col, vdim - 4));
    if constexpr (VALUES == kWords) {
        const uint32_t c = min(col, vdim - 4);
        uint64_t x;                                            // (two-byte aligned)
        __builtin_memcpy(&x, reinterpret_cast<const char*>(base) + (row_offset + 2 * c), 8);
        x >>= 16 * ((col - c) & 3);
        return make_uint2((uint32_t)x, (uint32_t)(x >> 32));
    }
    const uint32_t last = vdim - 1;
    auto one = [&](uint32_t j) { return (uint32_t)at<uint16_t>(base, row_offset + 2 * min(col + j, last)); };
    return make_uint2(one(0) | one(1) << 16, one(2) | one(3) << 16);
}

// The matrix products below contract over rows, so an operand's eight values lie in eight rows.  A lane therefore loads a few
// neighbouring columns of eight rows and sorts them in registers: of columns 4 n .. 4 n + 3 of lane n each goes to a tile of its own.
// Nothing goes through LDS for that (as two-byte stores of a transposed tile it took most of the time).

// Rows of a chunk: 64 while those make no more than a workgroup per CU (256) in step 3, which then waits for one chain of a workgroup,
// half as long; else 128.  All three steps, chunks of 64 / 128 rows: 16 heads of 128 x 128, 64 rows 14.5 / 15.4 us, 128 rows 15.5 / 19.3, 512 rows
// 22.8 / 22.8, 2048 rows 45.6 / 36.3; 4 heads of 64 x 64, 512 rows 12.5 / 16.4, 2048 rows 16.8 / 18.2; selective, 32 heads, 512 rows
// 26.6 / 28.9, 2048 rows 49.7 / 42.0.
uint32_t short_chunks(uint32_t heads, uint32_t vdim) { return (uint32_t)(256 / std::max<uint64_t>(1, (uint64_t)heads * ((vdim + 63) / 64))); }   // that many at most
uint32_t chunk_rows(uint32_t rows, uint32_t heads, uint32_t vdim) { return (rows + 63) / 64 <= short_chunks(heads, vdim) ? 64 : 128; }
size_t state_bytes(uint32_t chunks, uint32_t heads, uint32_t dim, uint32_t vdim) { return (size_t)chunks * heads * vdim * lh_linear_attention_padded_dim(dim) * 4; }
// The chunk for a workspace of `bytes`, which a caller may have sized for 128 rows.
uint32_t chunk_in(size_t bytes, uint32_t rows, uint32_t heads, uint32_t dim, uint32_t vdim) {
    return bytes < state_bytes((rows + 63) / 64, heads, dim, vdim) ? 128 : chunk_rows(rows, heads, vdim);
}

// Step 1.  A wave takes 32 key columns and 64 value columns of one chunk of one head.  Row operand = decayed keys, column operand
// = values.  What binds is the split of the decayed keys (7 vector instructions a value) and the latency of the loads.
// 2048 rows, 16 heads of 128 x 128: 24.5 -> 13 us (64 key columns a wave: 16, half as many waves to hide the loads).
template <int DQ, uint32_t CHUNK, bool SELECTIVE, Values VALUES>
__global__ __launch_bounds__(256) void chunk_state_kernel(const ChunkArgs a) {
    __shared__ float decays[4][CHUNK];                         // [wave][row]: from the row to its half's end
    const uint32_t lane = threadIdx.x & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), n = lane & 15, g = lane >> 4;
    constexpr uint32_t kblocks = DQ / 32;
    const uint32_t vtiles = (a.vdim + 63) / 64, unit = blockIdx.x * 4 + wave;
    const bool on = unit < kblocks * vtiles * a.heads * a.chunks;
    const uint32_t kb = unit % kblocks, r0 = unit / kblocks, vb = r0 % vtiles, h = (r0 / vtiles) % a.heads, c = on ? r0 / (vtiles * a.heads) : 0;
    const uint32_t t0 = c * CHUNK, L = min(CHUNK, a.rows - t0);
    const uint32_t kstride = a.key_heads * DQ * 2, vstride = a.heads * a.vdim * 2, kcol = kb * 32 + n * 2, vcol = vb * 64 + n * 4;   // strides in bytes
    const uint16_t *kp = a.k + ((size_t)t0 * a.key_heads + h / (a.heads / a.key_heads)) * DQ, *vp = a.v + ((size_t)t0 * a.heads + h) * a.vdim;
    struct Rows { uint32_t k[8]; uint2 v[8]; } rows[CHUNK / 32];
    const uint32_t k0 = 8 * g * kstride, v0 = 8 * g * vstride;
    auto fetch = [&](Rows& to, uint32_t s0) {                  // (rows past the last: the last again, whose decay is 0 then)
#pragma unroll
        for (uint32_t i = 0; i < 8; i++) {
            to.k[i] = at<uint32_t>(kp, min(k0 + (s0 + i) * kstride, (L - 1) * kstride) + 2 * kcol);
            to.v[i] = load_values<VALUES>(vp, min(v0 + (s0 + i) * vstride, (L - 1) * vstride), vcol, a.vdim);
        }
    };
    fetch(rows[0], 0);
    fetch(rows[1], 32);
    const float *pw = SELECTIVE ? nullptr : a.powers + h * (kHalf + 1), *sums = SELECTIVE ? a.sums + ((size_t)h * a.halves + CHUNK / kHalf * c) * kHalf : nullptr;
#pragma unroll
    for (uint32_t half = 0; half < CHUNK / kHalf; half++) {
        const uint32_t s = half * kHalf + lane, r = min(s, L - 1), end = min((half + 1) * kHalf, L) - 1;   // (a half without rows: its end is before them)
        float p;
        if constexpr (SELECTIVE) p = expf(sums[end] - sums[r]) * a.sizes[((size_t)h * a.halves + CHUNK / kHalf * c) * kHalf + r];
        else p = pw[end - r];
        decays[wave][s] = s < L ? p : 0.0f;
    }
    const float to_end = L <= kHalf ? 1.0f : SELECTIVE ? expf(sums[L - 1]) : pw[L - kHalf];   // from the first half's end to the chunk's
    __syncthreads();
    if (!on) return;
    const uint32_t keep = (kcol < a.dim ? 0xFFFFu : 0u) | (kcol + 1 < a.dim ? 0xFFFF0000u : 0u);   // key columns that exist
    lh_f32x4 acc[2][4];
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int d = 0; d < 4; d++) acc[j][d] = (lh_f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (uint32_t step = 0; step < CHUNK / 32; step++) {
        const uint32_t s0 = step * 32;
        if (s0 >= L) break;
        const Rows& now = rows[step];
        if (step + 2 < CHUNK / 32) fetch(rows[step + 2], s0 + 64);
        if (s0 == kHalf)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int d = 0; d < 4; d++) acc[j][d] *= to_end;
        lh_bf16x8 vf[4];
#pragma unroll
        for (int d = 0; d < 4; d++) {
            uint32_t w[4];
#pragma unroll
            for (int i = 0; i < 4; i++) w[i] = pick(now.v[2 * i], now.v[2 * i + 1], d);
            vf[d] = bf8(w);
        }
        float p[8];
#pragma unroll
        for (int i = 0; i < 8; i++) p[i] = decays[wave][s0 + 8 * g + i];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            uint32_t w[3][4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float f[2];
#pragma unroll
                for (int b = 0; b < 2; b++) {
                    const uint32_t x = now.k[2 * i + b] & keep;
                    f[b] = __builtin_bit_cast(float, j ? x & 0xFFFF0000u : x << 16) * p[2 * i + b];
                }
                split3_pair(f[0], f[1], w[0][i], w[1][i], w[2][i]);
            }
#pragma unroll
            for (int d = 0; d < 4; d++)
#pragma unroll
                for (int z = 0; z < 3; z++) acc[j][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf8(w[z]), vf[d], acc[j][d], 0, 0, 0);
        }
    }
    // a lane holds eight neighbouring key columns of four value columns
    float* U = a.chunk_state + ((size_t)c * a.heads + h) * a.vdim * DQ + kb * 32 + g * 8;
#pragma unroll
    for (int d = 0; d < 4; d++) {
        if (vcol + d >= a.vdim) continue;
        float4* to = reinterpret_cast<float4*>(U + (size_t)(vcol + d) * DQ);
#pragma unroll
        for (int i = 0; i < 2; i++) to[i] = make_float4(acc[0][d][2 * i], acc[1][d][2 * i], acc[0][d][2 * i + 1], acc[1][d][2 * i + 1]);
    }
}

// Step 2.  A thread owns four neighbouring state values and walks the chunks, eight loads ahead.  Memory binds: 15 -> 8 us for 2048
// rows, 16 heads of 128 x 128, with half as many states.
template <bool SELECTIVE>
__global__ __launch_bounds__(256) void chunk_scan_kernel(const ChunkArgs a, uint32_t dq) {
    const size_t per_head4 = (size_t)a.vdim * dq / 4, total4 = per_head4 * a.heads, i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= total4) return;
    const uint32_t h = (uint32_t)(i / per_head4);
    const float* pw = SELECTIVE ? nullptr : a.powers + h * (kHalf + 1);
    float4* st = reinterpret_cast<float4*>(a.state) + i;
    float4* u = reinterpret_cast<float4*>(a.chunk_state) + i;
    float4 s = *st;
    constexpr uint32_t P = 8;
    for (uint32_t c0 = 0; c0 < a.chunks; c0 += P) {
        float4 x[P];
        float d[P], d2[P];                                     // selective: the logarithm; else the decays of the two halves
#pragma unroll
        for (uint32_t j = 0; j < P; j++) {
            const uint32_t c = min(c0 + j, a.chunks - 1), L = min(a.chunk, a.rows - c * a.chunk);
            x[j] = u[(size_t)c * total4];
            if constexpr (SELECTIVE) {
                const float* sums = a.sums + ((size_t)h * a.halves + a.chunk / kHalf * c) * kHalf;
                d[j] = sums[min(L, kHalf) - 1] + (L > kHalf ? sums[L - 1] : 0.0f);
            } else { d[j] = pw[min(L, kHalf)]; d2[j] = pw[L - min(L, kHalf)]; }
        }
#pragma unroll
        for (uint32_t j = 0; j < P; j++) {
            if (c0 + j >= a.chunks) break;
            u[(size_t)(c0 + j) * total4] = s;
            const float f = SELECTIVE ? expf(d[j]) : d[j];
            if constexpr (!SELECTIVE) { s.x *= d2[j]; s.y *= d2[j]; s.z *= d2[j]; s.w *= d2[j]; }
            s.x = __builtin_fmaf(f, s.x, x[j].x); s.y = __builtin_fmaf(f, s.y, x[j].y);
            s.z = __builtin_fmaf(f, s.z, x[j].z); s.w = __builtin_fmaf(f, s.w, x[j].w);
        }
    }
    *st = s;
}

// Step 3.  A workgroup takes one chunk of one head and 64 value columns; a wave 32 of its rows.
// Scores transposed (row operand keys, column operand queries), so that the decayed scores are in operand order for
// O^T = V^T P^T, whose k index 8g + j is row 4g + j of the first 16-row tile (j < 4) or 4g + j - 4 of the second.
// The state is split into its bf16 terms once, by all waves, into LDS in operand order.  (Every wave of a chunk of 64 rows splitting
// it for itself was what bound this step: twice the states, four times the splits.)  What binds now is the vector work on the
// scores, so the operands of keys and values serve 32 rows.  2048 rows, 16 heads of 128 x 128:
// 32 -> 20.5 us.
template <int DQ, uint32_t CHUNK, bool SELECTIVE, Values VALUES>
__global__ __launch_bounds__(256, DQ <= 64 ? 3 : DQ <= 128 ? 2 : 1) void chunk_output_kernel(const ChunkArgs a) {
    constexpr int KB = DQ < 128 ? DQ : 128;                    // key columns of the state in LDS at a time
    constexpr int NB = CHUNK / 64;                             // blocks of 16 rows a wave takes
    __shared__ uint4 terms[3][4][KB / 32][64];                 // [term][value tile][32 key columns][lane]
    __shared__ float pws[SELECTIVE ? CHUNK : kHalf + 4], sizes[SELECTIVE ? CHUNK : 1];   // powers of the decay, or running sums of its logarithm
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6)), g = lane >> 4, n = lane & 15;
    const uint32_t vtiles = (a.vdim + 63) / 64, vb = blockIdx.x % vtiles, h = (blockIdx.x / vtiles) % a.heads, c = blockIdx.x / (vtiles * a.heads);
    const uint32_t t0 = c * CHUNK, L = min(CHUNK, a.rows - t0), v0 = vb * 64;
    // late rows see more of the chunk: of two workgroups on a CU one has them on the SIMDs where the other has the early ones
    const uint32_t w0 = ((blockIdx.x >> 8) & 1 ? 3 - wave : wave) * (16 * NB);
    const bool on = w0 < L;
    const uint32_t kh = h / (a.heads / a.key_heads), kstride = a.key_heads * DQ * 2, vstride = a.heads * a.vdim * 2;   // strides in bytes
    const uint16_t *qp = a.q + ((size_t)t0 * a.key_heads + kh) * DQ, *kp = a.k + ((size_t)t0 * a.key_heads + kh) * DQ, *vp = a.v + ((size_t)t0 * a.heads + h) * a.vdim;
    const float* S = a.chunk_state + (((size_t)c * a.heads + h) * a.vdim + v0) * DQ;
    constexpr uint32_t each = 4 * (KB / 32) * 64 / 256;        // operands of eight values a thread brings in
    float4 x[each][2];
    auto fetch_state = [&](uint32_t k0) {
#pragma unroll
        for (uint32_t e = 0; e < each; e++) {
            const uint32_t u = tid + 256 * e, l = u & 63, i = (u >> 6) % (KB / 32), d = (u >> 6) / (KB / 32);
            const uint32_t o = (min((l & 15) * 4 + d, a.vdim - 1 - v0) * DQ + k0 + i * 32 + (l >> 4) * 8) * 4;
            x[e][0] = at<float4>(S, o);
            x[e][1] = at<float4>(S, o + 16);
        }
    };
    fetch_state(0);
    lh_bf16x8 qf[NB][DQ / 32];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int i = 0; i < DQ / 32; i++) qf[b][i] = at<lh_bf16x8>(qp, min(w0 + 16 * b + n, L - 1) * kstride + i * 64 + g * 16);
    struct Rows { lh_bf16x8 k[2][DQ / 32]; uint2 v[8]; } next;
    auto fetch = [&](uint32_t s0) {                            // 32 rows of keys and values, in operand order
#pragma unroll
        for (uint32_t u = 0; u < 2; u++) {
            const uint32_t o = min(n * kstride + (s0 + u * 16) * kstride, (L - 1) * kstride) + g * 16;
#pragma unroll
            for (int i = 0; i < DQ / 32; i++) next.k[u][i] = at<lh_bf16x8>(kp, o + i * 64);
        }
#pragma unroll
        for (uint32_t i = 0; i < 8; i++)
            next.v[i] = load_values<VALUES>(vp, min(4 * g * vstride + (s0 + (i >> 2) * 16 + (i & 3)) * vstride, (L - 1) * vstride), v0 + n * 4, a.vdim);
    };
    fetch(0);
    if constexpr (SELECTIVE) {
        if (tid < CHUNK) {
            const size_t i = ((size_t)h * a.halves + CHUNK / kHalf * c) * kHalf + min(tid, L - 1);
            pws[tid] = a.sums[i];
            sizes[tid] = a.sizes[i];
        }
    } else if (tid <= kHalf) pws[tid] = a.powers[h * (kHalf + 1) + tid];
    if (a.dim != DQ) {                                         // columns that do not exist
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int i = 0; i < DQ / 32; i++)
#pragma unroll
                for (uint32_t j = 0; j < 8; j++) if (i * 32 + g * 8 + j >= a.dim) qf[b][i][j] = (__bf16)0.0f;
    }
    lh_f32x4 o[NB][4];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int d = 0; d < 4; d++) o[b][d] = (lh_f32x4){0.f, 0.f, 0.f, 0.f};
    // the state's part, decayed afterwards
#pragma unroll
    for (int k0 = 0; k0 < DQ; k0 += KB) {
        if (k0) { __syncthreads(); fetch_state(k0); }
#pragma unroll
        for (uint32_t e = 0; e < each; e++) {
            const float f[8] = {x[e][0].x, x[e][0].y, x[e][0].z, x[e][0].w, x[e][1].x, x[e][1].y, x[e][1].z, x[e][1].w};
            uint32_t p[3][4];
#pragma unroll
            for (int j = 0; j < 4; j++) split3_pair(f[2 * j], f[2 * j + 1], p[0][j], p[1][j], p[2][j]);
#pragma unroll
            for (int z = 0; z < 3; z++) (&terms[z][0][0][0])[tid + 256 * e] = make_uint4(p[z][0], p[z][1], p[z][2], p[z][3]);
        }
        __syncthreads();
        if (!on) continue;
        // (the small terms of all columns first: the large ones are then rounded once a product, not with each of their remainders as well)
#pragma unroll
        for (int z = 2; z >= 0; z--)
#pragma unroll
            for (int i = 0; i < KB / 32; i++) {
                lh_bf16x8 sf[4];
#pragma unroll
                for (int d = 0; d < 4; d++) sf[d] = __builtin_bit_cast(lh_bf16x8, terms[z][d][i][lane]);
#pragma unroll
                for (int b = 0; b < NB; b++)
#pragma unroll
                    for (int d = 0; d < 4; d++) o[b][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(sf[d], qf[b][k0 / 32 + i], o[b][d], 0, 0, 0);
            }
    }
    if (!on) return;
    // Rows of the second half: what they take from before it is decayed to the first half's end as it comes, and from there when their
    // own half begins.
    const uint32_t half0 = CHUNK > kHalf && w0 >= kHalf ? kHalf : 0;
    const float half_end = SELECTIVE ? pws[kHalf - 1] : 0.0f;
    if (half0) {
        const float f = SELECTIVE ? expf(half_end) : pws[kHalf];
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int d = 0; d < 4; d++) o[b][d] *= f;
    }
    float sum_to[NB];                                          // selective: the running sum at the half's end, then at the lane's row
#pragma unroll
    for (int b = 0; b < NB; b++) sum_to[b] = half_end;
    // the chunk's own rows, 32 at a time
#pragma unroll 1
    for (uint32_t s0 = 0; s0 <= w0; s0 += 32) {
        lh_f32x4 sc[NB][2];
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int u = 0; u < 2; u++) {
                sc[b][u] = (lh_f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < DQ / 32; i++) sc[b][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(next.k[u][i], qf[b][i], sc[b][u], 0, 0, 0);
            }
        lh_bf16x8 vf[4];
#pragma unroll
        for (int d = 0; d < 4; d++) {
            uint32_t w[4];
#pragma unroll
            for (int i = 0; i < 4; i++) w[i] = pick(next.v[2 * i], next.v[2 * i + 1], d);
            vf[d] = bf8(w);
        }
        if (s0 + 32 <= w0) fetch(s0 + 32);
        const bool across = s0 < half0;
        if (s0 == half0)
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const uint32_t tr = min(w0 + 16 * b + n, L - 1);
                sum_to[b] = pws[SELECTIVE ? tr : 0];
                const float f = SELECTIVE ? expf(sum_to[b]) : pws[tr - half0 + 1];
#pragma unroll
                for (int d = 0; d < 4; d++) o[b][d] *= f;
            }
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const uint32_t t = w0 + 16 * b + n, to = across ? kHalf - 1 : t;
            uint32_t p[3][4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float e[2];
#pragma unroll
                for (int y = 0; y < 2; y++) {
                    const int m = 2 * j + y;
                    const uint32_t s = s0 + (m >> 2) * 16 + g * 4 + (m & 3);
                    const float f = SELECTIVE ? expf(fminf(sum_to[b] - pws[s], 0.0f)) * sizes[s] : pws[min(to - s, kHalf)];
                    // the product is made for rows after t as well (skipping it would take a branch for each) and left out whatever it is:
                    // a step size or a power there may be no finite number
                    const float x = sc[b][m >> 2][m & 3] * f;
                    e[y] = s <= t ? x : 0.0f;
                }
                split3_pair(e[0], e[1], p[0][j], p[1][j], p[2][j]);
            }
            // (a sum of its own for these rows: what was added up before is rounded once for them, not with each term)
#pragma unroll
            for (int d = 0; d < 4; d++) {
                lh_f32x4 r = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[d], bf8(p[2]), (lh_f32x4){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                r = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[d], bf8(p[1]), r, 0, 0, 0);
                r = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[d], bf8(p[0]), r, 0, 0, 0);
                o[b][d] += r;
            }
        }
    }
    // a lane holds 16 neighbouring value columns of its rows
    const float skip = SELECTIVE ? a.skip[h] : 0.0f;
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const uint32_t t = w0 + 16 * b + n;
        if (t >= L) continue;
        float* out = a.out + ((size_t)(t0 + t) * a.heads + h) * a.vdim;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const uint32_t col = v0 + g * 16 + r * 4;
            if (col >= a.vdim) continue;
            float y[4];
            if constexpr (SELECTIVE) {
                const uint2 z = load_values<VALUES>(vp, t * vstride, col, a.vdim);
                y[0] = __builtin_bit_cast(float, z.x << 16); y[1] = __builtin_bit_cast(float, z.x & 0xFFFF0000u);
                y[2] = __builtin_bit_cast(float, z.y << 16); y[3] = __builtin_bit_cast(float, z.y & 0xFFFF0000u);
            }
#pragma unroll
            for (int d = 0; d < 4; d++) y[d] = SELECTIVE ? __builtin_fmaf(skip, y[d], o[b][d][r]) : o[b][d][r] * a.scale;
            if constexpr (VALUES == kPieces) *reinterpret_cast<float4*>(out + col) = make_float4(y[0], y[1], y[2], y[3]);
            else
#pragma unroll
                for (uint32_t d = 0; d < 4; d++) if (col + d < a.vdim) out[col + d] = y[d];
        }
    }
}

template <int DQ, uint32_t CHUNK, bool SELECTIVE, Values VALUES>
int launch_chunked(lh_context* ctx, const ChunkArgs& a, const char* op) {
    const uint32_t grid = a.chunks * a.heads * ((a.vdim + 63) / 64), waves = grid * (DQ / 32);
    hipLaunchKernelGGL((chunk_state_kernel<DQ, CHUNK, SELECTIVE, VALUES>), dim3((waves + 3) / 4), dim3(256), 0, ctx->stream, a);
    int r = lh_check_launch(op);
    if (r != LH_OK) return r;
    const size_t total4 = (size_t)a.heads * a.vdim * DQ / 4;
    hipLaunchKernelGGL((chunk_scan_kernel<SELECTIVE>), dim3((uint32_t)((total4 + 255) / 256)), dim3(256), 0, ctx->stream, a, (uint32_t)DQ);
    r = lh_check_launch(op);
    if (r != LH_OK) return r;
    hipLaunchKernelGGL((chunk_output_kernel<DQ, CHUNK, SELECTIVE, VALUES>), dim3(grid), dim3(256), 0, ctx->stream, a);
    return lh_check_launch(op);
}
template <uint32_t CHUNK, bool SELECTIVE, Values VALUES>
int launch_chunked_values(lh_context* ctx, const ChunkArgs& a, const char* op) {
    switch (lh_linear_attention_padded_dim(a.dim)) {
        case 32: return launch_chunked<32, CHUNK, SELECTIVE, VALUES>(ctx, a, op);
        case 64: return launch_chunked<64, CHUNK, SELECTIVE, VALUES>(ctx, a, op);
        case 128: return launch_chunked<128, CHUNK, SELECTIVE, VALUES>(ctx, a, op);
        default: return launch_chunked<256, CHUNK, SELECTIVE, VALUES>(ctx, a, op);
    }
}
template <uint32_t CHUNK, bool SELECTIVE>
int launch_chunked_rows(lh_context* ctx, const ChunkArgs& a, const char* op) {
    if (a.vdim % 4 == 0) return launch_chunked_values<CHUNK, SELECTIVE, kPieces>(ctx, a, op);
    return a.vdim > 4 ? launch_chunked_values<CHUNK, SELECTIVE, kWords>(ctx, a, op) : launch_chunked_values<CHUNK, SELECTIVE, kSingles>(ctx, a, op);
}
template <bool SELECTIVE>
int launch_chunked_dim(lh_context* ctx, ChunkArgs& a, const char* op) {
    a.chunks = (a.rows + a.chunk - 1) / a.chunk;
    return a.chunk == 64 ? launch_chunked_rows<64, SELECTIVE>(ctx, a, op) : launch_chunked_rows<128, SELECTIVE>(ctx, a, op);
}

template <typename T, Decay DECAY>
int launch_recurrent(lh_context* ctx, const RecurrentArgs& a, const char* op) {
    const uint64_t grid = (uint64_t)a.heads * ((a.vdim + 15) / 16);
    LH_REQUIRE(grid < 0x7FFFFFFFull, "%s: heads %u, vdim %u", op, a.heads, a.vdim);
    const bool whole = (((uintptr_t)a.q | (uintptr_t)a.k) & 15) == 0;          // (a row's keys and queries start at multiples of 32 values)
    const uint64_t columns = (uint64_t)a.heads * a.vdim;
    // A wave a column from 65 key columns on (below, half its lanes would have none): few rows always (us of 1, 2 and 7 rows of 16 heads, bf16, then so: 128 x 128 5.4,
    // 6.4, 12.1 and 4.8, 4.6, 4.9; 256 x 128 10.7, 14.6, 33.2 and 4.7, 4.6, 4.8), and of many rows where a lane of the other form would hold
    // more than eight 32-bit values or compute the rows' steps (200 rows of 48 heads, f32: 256 x 128 189 and 99, selective 128 x 128 186 and 98);
    // else up to two waves a SIMD (128 x 128, 8, 16 and 24 heads: 39, 40, 40 and 21, 33, 47), of bf16 with 129 to 256 key columns, whose two values share a
    // register there, up to five (200 rows of 256 x 128 with 32, 40, 48 and 64 heads: 66, 88, 88 and 88 us, and 63, 78, 91 and 119).
    const uint64_t cus = (uint64_t)ctx->cu_count;
    const bool few = a.rows < 8, wide = few || DECAY == kSelective || (a.dq <= 128 ? columns <= 8 * cus : sizeof(T) == 4 || a.dq > 256 || columns <= 20 * cus);
    if (whole && a.dq > 64 && a.dq <= 512 && wide) {
        const dim3 blocks((uint32_t)((columns + 3) / 4));
#define LH_REC(NR_, AHEAD_) hipLaunchKernelGGL((recurrent_wide_kernel<T, NR_, AHEAD_, DECAY>), blocks, dim3(256), 0, ctx->stream, a)
        // What is requested ahead past the last row is traffic for nothing, so that few rows have fewer ahead (selective 128 x 128, 128 heads, f32: 8 rows
        // 27.4 us with sixteen ahead, 20.5 with twelve; 16 rows 45.6, with eight 32.1; 64 rows 99.6, 85.6; bf16 20.0, 16.8; 30.3, 28.3; 73.1, 75.7).
        if (a.dq <= 128) { if (few) LH_REC(2, 4); else if (a.rows < 12) LH_REC(2, 12); else if (a.rows < 24) LH_REC(2, 8); else LH_REC(2, 16); }
        else if (a.dq <= 256) { if (few) LH_REC(4, 4); else if (a.rows < 12 && sizeof(T) == 2) LH_REC(4, 12); else LH_REC(4, 8); }
        else LH_REC(8, 4);
#undef LH_REC
        return lh_check_launch(op);
    }
    if (a.rows >= 8 && whole) {
#define LH_REC(NR_, AHEAD_) hipLaunchKernelGGL((recurrent_rows_kernel<T, NR_, AHEAD_, DECAY>), dim3((uint32_t)grid), dim3(256), 0, ctx->stream, a)
        if (a.dq <= 32) LH_REC(2, 8);
        else if (a.dq <= 64) LH_REC(4, 8);
        else if (a.dq <= 128) { if constexpr (DECAY != kSelective) LH_REC(8, 8); }
        else if (a.dq <= 256) { if constexpr (DECAY != kSelective && sizeof(T) == 2) LH_REC(16, 4); }
        else LH_REC(64, 1);
#undef LH_REC
        return lh_check_launch(op);
    }
#define LH_REC(NR_) hipLaunchKernelGGL((recurrent_kernel<T, NR_, DECAY>), dim3((uint32_t)grid), dim3(256), 0, ctx->stream, a)
    if (a.dq <= 32) LH_REC(2);
    else if (a.dq <= 64) LH_REC(4);
    else if (a.dq <= 128) LH_REC(8);
    else if (a.dq <= 256) LH_REC(16);
    else if (a.dq <= 512) LH_REC(32);
    else LH_REC(64);
#undef LH_REC
    return lh_check_launch(op);
}

// The chunk kernels address the rows of a chunk with 32-bit byte offsets.  Rows of 2^24 values and more (32 MB each) walk the recurrence:
// their columns alone fill the chip.
bool chunk_offsets_fit(uint32_t heads, uint32_t dq, uint32_t vdim) { return (uint64_t)heads * std::max(dq, vdim) < (1u << 24); }

}  // namespace

extern "C" {

uint32_t lh_linear_attention_padded_dim(uint32_t dim) { return dim <= 32 ? 32u : dim <= 64 ? 64u : (dim + 127) / 128 * 128; }

// (what is enough for `rows` is enough for fewer)
size_t lh_linear_attention_workspace_bytes(uint32_t rows, uint32_t heads, uint32_t dim, uint32_t vdim) {
    return state_bytes(std::max((rows + 127) / 128, std::min((rows + 63) / 64, short_chunks(heads, vdim))), heads, dim, vdim);
}

int lh_linear_attention_recurrent_into(lh_batch* batch, const lh_buffer* q, const lh_buffer* k, const lh_buffer* v, int dtype, lh_buffer* state,
                                       const lh_buffer* decay, lh_buffer* output, uint32_t rows, uint32_t heads, uint32_t dim, uint32_t vdim, float scale) {
    const char* op = "linear_attention_recurrent";
    LH_REQUIRE(batch, "%s: batch is null", op);
    LH_REQUIRE(dtype == LH_F32 || dtype == LH_BF16, "%s: dtype %d", op, dtype);
    LH_REQUIRE(heads > 0 && dim > 0 && dim <= 1024 && vdim > 0, "%s: heads %u, dim %u, vdim %u", op, heads, dim, vdim);
    if (rows == 0) return LH_OK;
    const uint32_t dq = lh_linear_attention_padded_dim(dim);
    const size_t es = dtype == LH_F32 ? 4 : 2;
    LH_NEED(q, (size_t)rows * heads * dq * es, op, "q");
    LH_NEED(k, (size_t)rows * heads * dq * es, op, "k");
    LH_NEED(v, (size_t)rows * heads * vdim * es, op, "v");
    LH_NEED(state, (size_t)heads * vdim * dq * 4, op, "state");
    LH_NEED(decay, (size_t)heads * 4, op, "decay");
    LH_NEED(output, (size_t)rows * heads * vdim * 4, op, "output");
    RecurrentArgs a{};
    a.q = q->ptr; a.k = k->ptr; a.v = v->ptr; a.state = (float*)state->ptr; a.decay = (const float*)decay->ptr; a.out = (float*)output->ptr;
    a.rows = rows; a.heads = a.key_heads = heads; a.dim = dim; a.dq = dq; a.vdim = vdim; a.scale = scale;
    const int r = dtype == LH_F32 ? launch_recurrent<float, kFixed>(batch->ctx, a, op) : launch_recurrent<uint16_t, kFixed>(batch->ctx, a, op);
    if (r == LH_OK) batch->dispatch_count++;
    return r;
}

int lh_linear_attention_chunked_into(lh_batch* batch, const lh_buffer* q, const lh_buffer* k, const lh_buffer* v, lh_buffer* state,
                                     const lh_buffer* decay_powers, lh_buffer* workspace, lh_buffer* output, uint32_t rows, uint32_t heads, uint32_t dim,
                                     uint32_t vdim, float scale) {
    const char* op = "linear_attention_chunked";
    LH_REQUIRE(batch, "%s: batch is null", op);
    LH_REQUIRE(heads > 0 && dim > 0 && dim <= 256 && vdim > 0, "%s: heads %u, dim %u, vdim %u", op, heads, dim, vdim);
    if (rows == 0) return LH_OK;
    const uint32_t dq = lh_linear_attention_padded_dim(dim);
    LH_NEED(q, (size_t)rows * heads * dq * 2, op, "q");
    LH_NEED(k, (size_t)rows * heads * dq * 2, op, "k");
    LH_NEED(v, (size_t)rows * heads * vdim * 2, op, "v");
    LH_NEED(state, (size_t)heads * vdim * dq * 4, op, "state");
    LH_NEED(decay_powers, (size_t)heads * (kHalf + 1) * 4, op, "decay_powers");
    LH_NEED(workspace, state_bytes((rows + 127) / 128, heads, dim, vdim), op, "workspace");
    LH_NEED(output, (size_t)rows * heads * vdim * 4, op, "output");
    LH_REQUIRE((((uintptr_t)q->ptr | (uintptr_t)k->ptr | (uintptr_t)v->ptr | (uintptr_t)state->ptr | (uintptr_t)workspace->ptr | (uintptr_t)output->ptr) & 15) == 0,
               "%s: buffers must be 16-byte aligned", op);
    if (!chunk_offsets_fit(heads, dq, vdim)) {
        RecurrentArgs r{};
        r.q = q->ptr; r.k = k->ptr; r.v = v->ptr; r.state = (float*)state->ptr; r.out = (float*)output->ptr;
        r.decay = (const float*)decay_powers->ptr + 1;
        r.rows = rows; r.heads = r.key_heads = heads; r.dim = dim; r.dq = dq; r.vdim = vdim; r.scale = scale;
        const int rc = launch_recurrent<uint16_t, kPowers>(batch->ctx, r, op);
        if (rc == LH_OK) batch->dispatch_count++;
        return rc;
    }
    ChunkArgs a{};
    a.q = (const uint16_t*)q->ptr; a.k = (const uint16_t*)k->ptr; a.v = (const uint16_t*)v->ptr; a.state = (float*)state->ptr;
    a.powers = (const float*)decay_powers->ptr; a.chunk_state = (float*)workspace->ptr; a.out = (float*)output->ptr;
    a.rows = rows; a.heads = a.key_heads = heads; a.dim = dim; a.vdim = vdim; a.chunk = chunk_in(workspace->len, rows, heads, dim, vdim); a.halves = (rows + kHalf - 1) / kHalf; a.scale = scale;
    LH_REQUIRE((uint64_t)((rows + 63) / 64) * heads * ((vdim + 63) / 64) * 8 < 0x7FFFFFFFull, "%s: %u rows", op, rows);
    const int r = launch_chunked_dim<false>(batch->ctx, a, op);
    if (r == LH_OK) batch->dispatch_count += 3;
    return r;
}

// [heads][halves][64] running sums, then as many step sizes
size_t lh_selective_steps_bytes(uint32_t rows, uint32_t heads) { return (size_t)((rows + kHalf - 1) / kHalf) * kHalf * heads * 2 * 4; }

int lh_selective_recurrent_into(lh_batch* batch, const lh_buffer* x, const lh_buffer* b, const lh_buffer* c, int dtype, const lh_buffer* dt_raw,
                                const lh_buffer* dt_bias, const lh_buffer* a_log, const lh_buffer* skip, lh_buffer* memory, lh_buffer* output, uint32_t rows,
                                uint32_t heads, uint32_t vdim, uint32_t groups, uint32_t state) {
    const char* op = "selective_recurrent";
    LH_REQUIRE(batch, "%s: batch is null", op);
    LH_REQUIRE(dtype == LH_F32 || dtype == LH_BF16, "%s: dtype %d", op, dtype);
    LH_REQUIRE(heads > 0 && groups > 0 && heads % groups == 0 && state > 0 && state <= 1024 && vdim > 0, "%s: heads %u over %u groups, state %u, vdim %u", op, heads,
               groups, state, vdim);
    if (rows == 0) return LH_OK;
    const uint32_t dq = lh_linear_attention_padded_dim(state);
    const size_t es = dtype == LH_F32 ? 4 : 2;
    LH_NEED(x, (size_t)rows * heads * vdim * es, op, "x");
    LH_NEED(b, (size_t)rows * groups * dq * es, op, "b");
    LH_NEED(c, (size_t)rows * groups * dq * es, op, "c");
    LH_NEED(dt_raw, (size_t)rows * heads * 4, op, "dt_raw");
    LH_NEED(dt_bias, (size_t)heads * 4, op, "dt_bias");
    LH_NEED(a_log, (size_t)heads * 4, op, "a_log");
    LH_NEED(skip, (size_t)heads * 4, op, "skip");
    LH_NEED(memory, (size_t)heads * vdim * dq * 4, op, "memory");
    LH_NEED(output, (size_t)rows * heads * vdim * 4, op, "output");
    RecurrentArgs a{};
    a.q = c->ptr; a.k = b->ptr; a.v = x->ptr; a.state = (float*)memory->ptr; a.out = (float*)output->ptr;
    a.dt_raw = (const float*)dt_raw->ptr; a.dt_bias = (const float*)dt_bias->ptr; a.a_log = (const float*)a_log->ptr; a.skip = (const float*)skip->ptr;
    a.rows = rows; a.heads = heads; a.key_heads = groups; a.dim = state; a.dq = dq; a.vdim = vdim; a.scale = 1.0f;
    const int r = dtype == LH_F32 ? launch_recurrent<float, kSelective>(batch->ctx, a, op) : launch_recurrent<uint16_t, kSelective>(batch->ctx, a, op);
    if (r == LH_OK) batch->dispatch_count++;
    return r;
}

int lh_selective_chunked_into(lh_batch* batch, const lh_buffer* x, const lh_buffer* b, const lh_buffer* c, const lh_buffer* dt_raw, const lh_buffer* dt_bias,
                              const lh_buffer* a_log, const lh_buffer* skip, lh_buffer* memory, lh_buffer* steps, lh_buffer* workspace, lh_buffer* output,
                              uint32_t rows, uint32_t heads, uint32_t vdim, uint32_t groups, uint32_t state) {
    const char* op = "selective_chunked";
    LH_REQUIRE(batch, "%s: batch is null", op);
    LH_REQUIRE(heads > 0 && groups > 0 && heads % groups == 0 && state > 0 && state <= 256 && vdim > 0, "%s: heads %u over %u groups, state %u, vdim %u", op, heads,
               groups, state, vdim);
    if (rows == 0) return LH_OK;
    const uint32_t dq = lh_linear_attention_padded_dim(state);
    LH_NEED(x, (size_t)rows * heads * vdim * 2, op, "x");
    LH_NEED(b, (size_t)rows * groups * dq * 2, op, "b");
    LH_NEED(c, (size_t)rows * groups * dq * 2, op, "c");
    LH_NEED(dt_raw, (size_t)rows * heads * 4, op, "dt_raw");
    LH_NEED(dt_bias, (size_t)heads * 4, op, "dt_bias");
    LH_NEED(a_log, (size_t)heads * 4, op, "a_log");
    LH_NEED(skip, (size_t)heads * 4, op, "skip");
    LH_NEED(memory, (size_t)heads * vdim * dq * 4, op, "memory");
    LH_NEED(steps, lh_selective_steps_bytes(rows, heads), op, "steps");
    LH_NEED(workspace, state_bytes((rows + 127) / 128, heads, state, vdim), op, "workspace");
    LH_NEED(output, (size_t)rows * heads * vdim * 4, op, "output");
    LH_REQUIRE((((uintptr_t)x->ptr | (uintptr_t)b->ptr | (uintptr_t)c->ptr | (uintptr_t)memory->ptr | (uintptr_t)workspace->ptr | (uintptr_t)output->ptr) & 15) == 0,
               "%s: buffers must be 16-byte aligned", op);
    if (!chunk_offsets_fit(heads, dq, vdim)) return lh_selective_recurrent_into(batch, x, b, c, LH_BF16, dt_raw, dt_bias, a_log, skip, memory, output, rows, heads, vdim, groups, state);
    ChunkArgs a{};
    a.q = (const uint16_t*)c->ptr; a.k = (const uint16_t*)b->ptr; a.v = (const uint16_t*)x->ptr; a.state = (float*)memory->ptr;
    a.chunk_state = (float*)workspace->ptr; a.out = (float*)output->ptr; a.skip = (const float*)skip->ptr;
    a.rows = rows; a.heads = heads; a.key_heads = groups; a.dim = state; a.vdim = vdim; a.chunk = chunk_in(workspace->len, rows, heads, state, vdim); a.halves = (rows + kHalf - 1) / kHalf; a.scale = 1.0f;
    LH_REQUIRE((uint64_t)((rows + 63) / 64) * heads * ((vdim + 63) / 64) * 8 < 0x7FFFFFFFull, "%s: %u rows", op, rows);
    float* sums = (float*)steps->ptr;
    float* sizes = sums + (size_t)a.halves * kHalf * heads;
    a.sums = sums; a.sizes = sizes;
    hipLaunchKernelGGL(chunk_steps_kernel, dim3(a.halves * heads), dim3(64), 0, batch->ctx->stream, (const float*)dt_raw->ptr, (const float*)dt_bias->ptr,
                       (const float*)a_log->ptr, sums, sizes, rows, heads, a.halves);
    int r = lh_check_launch(op);
    if (r == LH_OK) r = launch_chunked_dim<true>(batch->ctx, a, op);
    if (r == LH_OK) batch->dispatch_count += 4;
    return r;
}

}  // extern "C"
