// Causal softmax attention over bf16 (or f32) caches, with one or two score maps per head.  With two maps (differential
// attention) both share the head's values and are combined in the same kernel: the difference of the two averages, the
// second times lambda, an RMS norm over the head, a constant factor.
//
// Caches: keys [position][kv head][map][DQ], values in blocks of 32 positions [block][kv head][DV][32] whose 32 entries
// are in lh_block_slot order.  The queries of one kv head's group are packed: packed row r = query row r / R, head r % R of
// the group (R heads per kv head), so a tile of 16 packed rows uses the matrix cores fully also for one query row.
//
// Matrix-core form (bf16): a step of 32 keys computes S^T = K Q^T (two 16 x 16 tiles; lane = packed row (lane & 15), keys
// 4g .. 4g + 3 of each tile, g = lane >> 4), so a row's maximum and sum are eight registers and two lane exchanges, and
// the weights are already where O^T = V^T P^T wants them: its k index 8g + j is key 4g + j of tile 0 (j < 4) or key
// 4g + j - 4 of tile 1, which is the order of the value blocks.  Scores, weights and sums are f32; a weight enters the
// product as the sum of three bf16 terms, which is all of its 24 bits.
//   attention_tile_kernel   many rows: four waves share key and value blocks through LDS
//   attention_one_kernel    one row over a few hundred keys (one_blocks): one workgroup per kv head
//   attention_split_kernel  few rows: every wave walks its own share of the blocks straight from global memory; the
//                           workgroup's four partial results are merged in LDS, the workgroups' by attention_merge_kernel
//   attention_wide_kernel   f32 caches: f32 matrix instructions, 16 packed rows a workgroup
//   attention_vector_kernel f32 caches, a few rows: the vector ALU, a workgroup per row and head
// Plain form (any dtype, any dim): attention_plain_kernel, one workgroup per query row and head.
#include "softmax_attention.hpp"
#include <type_traits>

namespace {

// The B operand of S^T: query values of packed row `row` (zero past the rows and past dim).  (With the address as an argument, for attention_one_kernel to share
// it, attention_tile_kernel came out in another order of instructions: two maps of 64 and 128 columns, 8 heads, 512 rows at 1024 29.8 us, then 30.4.)
template <int DQ, int MAPS>
__device__ __forceinline__ void load_queries(lh_bf16x8 (&qf)[MAPS][DQ / 32], const AttentionArgs& a, uint32_t g, uint32_t row, uint32_t lane) {
    const uint32_t R = a.heads / a.kv_heads, t = row / R, h = g * R + (row - t * R);
    const bool on = t < a.rows;
#pragma unroll
    for (int mp = 0; mp < MAPS; mp++)
#pragma unroll
        for (int c = 0; c < DQ / 32; c++) {
            const uint32_t k = c * 32 + (lane >> 4) * 8;
            u32x4 v = {0u, 0u, 0u, 0u};
            if (on && k < a.dim) {
                v = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(a.q) + (((size_t)t * a.heads + h) * MAPS + mp) * DQ + k);
                if (!(a.scale > 0.0f)) {
#pragma unroll
                    for (int j = 0; j < 4; j++) v[j] = a.scale < 0.0f ? v[j] ^ 0x80008000u : 0u;      // (no number: scale2 is none either)
                }
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    if (k + 2 * j >= a.dim) v[j] = 0u;
                    else if (k + 2 * j + 1 >= a.dim) v[j] &= 0xFFFFu;
                }
            }
            qf[mp][c] = __builtin_bit_cast(lh_bf16x8, v);
        }
}

// A finished row: o[i][r] holds value 16 i + 4g + r of packed row (lane & 15), for every map unnormalised with sum l.
template <int DV, int MAPS>
__device__ __forceinline__ void finish_row(const AttentionArgs& a, lh_f32x4 (&o)[MAPS][DV / 16], const float (&l)[MAPS], float m0, uint32_t g, uint32_t row, uint32_t lane) {   // m0: the first map's maximum
    const uint32_t R = a.heads / a.kv_heads, t = row / R, h = g * R + (row - t * R);
    float inv[MAPS];
#pragma unroll
    for (int mp = 0; mp < MAPS; mp++) inv[mp] = 1.0f / l[mp];
    if (MAPS == 1 && a.sink) inv[0] = 1.0f / (l[0] + __builtin_amdgcn_exp2f(a.sink[h] * kLog2e - m0));
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < DV / 16; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            float v = o[0][i][r] * inv[0];
            if constexpr (MAPS == 2) v -= a.lambda * (o[MAPS - 1][i][r] * inv[MAPS - 1]);
            o[0][i][r] = v;
            if ((uint32_t)(i * 16 + (lane >> 4) * 4 + r) < a.vdim) ss += v * v;
        }
    float f = 1.0f;
    if constexpr (MAPS == 2) {
        ss = lh_column_sum(ss);
        f = rsqrtf(ss / (float)a.vdim + a.eps) * a.out_scale;
    }
    if (t >= a.rows) return;
    if (MAPS == 1 && a.gate) f = lh_sigmoid(a.gate[(size_t)t * a.heads + h]);
    uint16_t* out = static_cast<uint16_t*>(a.out) + ((size_t)t * a.heads + h) * a.vdim;
#pragma unroll
    for (int i = 0; i < DV / 16; i++) {
        const uint32_t c = i * 16 + (lane >> 4) * 4;
        if ((a.vdim & 3) == 0) {
            if (c < a.vdim) *reinterpret_cast<uint2*>(out + c) = make_uint2(lh_pack_bf(o[0][i][0] * f, o[0][i][1] * f), lh_pack_bf(o[0][i][2] * f, o[0][i][3] * f));
        } else {
#pragma unroll
            for (int r = 0; r < 4; r++) if (c + r < a.vdim) out[c + r] = lh_f2bf(o[0][i][r] * f);
        }
    }
}

typedef __attribute__((address_space(1))) const void gvoid;
typedef __attribute__((address_space(3))) void lvoid;

// 64 packed rows, 16 per wave; steps of 32 * NB keys through two LDS buffers.  A key row of the buffer is MAPS * DQ / 8 chunks
// of 16 bytes, chunk c at place c ^ (key & 7) (see linear_mfma_kernel for why and how); a column of a value block is four chunks, placed
// so that any eight or sixteen neighbouring columns read different banks.  With more than one split a workgroup takes its share of the key
// steps and leaves partial records.
// What binds is vector and matrix instructions at the clock that they leave (a step of 64 keys of two maps: 3600 cycles of matrix
// instructions per SIMD and about 3000 of vector instructions, before two values were rounded and reduced by one instruction each 5000:
// 2048 rows of 16 heads, two maps, at position 0 104 -> 95 us, at 2048 252 -> 216).  No product waits for the one before it: 95 -> 89.  With one map the two blocks of a step belong to two groups of four
// waves, whose sums meet at the end: 2048 rows of 16 heads of 192 and 128 columns 75 -> 61 us.  With two maps the registers do not suffice for that.
__device__ __forceinline__ uint32_t value_place(uint32_t col) { return ((col >> 2) & 1) * 2 + (((col >> 1) ^ (col >> 3)) & 1); }
template <int DQ, int DV, int MAPS, int NB, int G>
__global__ __launch_bounds__(256 * G, G == 2 ? 4 : MAPS * DV <= 256 ? 2 : 1) void attention_tile_kernel(const AttentionArgs a) {
    constexpr int KC = MAPS * DQ / 8, KCH = 32 * NB * KC, VB = DV * 4, VCH = NB * VB, T = 256 * G, NW = NB / G;   // chunks per key row; per step: keys, values
    constexpr uint32_t kSwizzle = KC >= 8 ? 7 : KC - 1;
    __shared__ uint4 sm[2][KCH + VCH];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), group = wave >> 2;
    const uint32_t R = a.heads / a.kv_heads, packed = a.rows * R, tiles = (packed + 63) / 64;
    // The long tiles first; where all workgroups are on the chip at once, two a CU, the second of a CU has as much less to do as the first
    // has more.
    const uint32_t order = blockIdx.x < a.resident || gridDim.x > 2 * a.resident ? blockIdx.x : gridDim.x - 1 - (blockIdx.x - a.resident);
    const uint32_t split = order % a.splits, gt = order / a.splits;
    const uint32_t g = gt % a.kv_heads, tile = tiles - 1 - gt / a.kv_heads;
    const uint32_t start = *a.position;
    const uint32_t row0 = tile * 64, row_last = min(row0 + 64, packed) - 1;
    const uint32_t last_key = min(start + row_last / R, a.capacity - 1), last_block = last_key / 32, nstep = last_block / NB + 1;
    const uint32_t per = (nstep + a.splits - 1) / a.splits, s0 = min(split * per, nstep), s1 = min(s0 + per, nstep);
    const uint32_t wrow = row0 + (wave & 3) * 16, row = wrow + (lane & 15);

    lh_bf16x8 qf[MAPS][DQ / 32];
    load_queries<DQ, MAPS>(qf, a, g, row, lane);
    const uint32_t limit = min(start + row / R, last_key), first_limit = start + wrow / R, wave_last = min(start + (wrow + 15) / R, last_key);
    lh_f32x4 o[MAPS][DV / 16];
    RowState st[MAPS];
#pragma unroll
    for (int mp = 0; mp < MAPS; mp++) {
        st[mp] = RowState{-INFINITY, 0.0f};
#pragma unroll
        for (int d = 0; d < DV / 16; d++) o[mp][d] = (lh_f32x4){0.f, 0.f, 0.f, 0.f};
    }

    const uint16_t* K = static_cast<const uint16_t*>(a.keys) + (size_t)g * MAPS * DQ;
    const uint16_t* V = static_cast<const uint16_t*>(a.values) + (size_t)g * DV * 32;
    const size_t krow = (size_t)a.kv_heads * MAPS * DQ, vblock = (size_t)a.kv_heads * DV * 32;
    auto load_step = [&](int buf, uint32_t s) {
#pragma unroll
        for (int i = 0; i < (KCH + T - 1) / T; i++) {
            if (KCH % T != 0 && i * T + wave * 64 >= KCH) break;                          // whole waves (KCH is a multiple of 64)
            const uint32_t c = i * T + tid, key = c / KC, ch = (c % KC) ^ (key & kSwizzle);
            const uint32_t p = min(s * (32 * NB) + key, last_key);                        // keys past the last are masked
            __builtin_amdgcn_global_load_lds((gvoid*)(K + p * krow + ch * 8), (lvoid*)&sm[buf][i * T + wave * 64], 16, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < (VCH + T - 1) / T; i++) {
            if (VCH % T != 0 && i * T + wave * 64 >= VCH) break;
            const uint32_t c = i * T + tid, e = c % VB, ch = (e & ~3u) | ((e & 3) ^ value_place(e >> 2));
            __builtin_amdgcn_global_load_lds((gvoid*)(V + min(s * NB + c / VB, last_block) * vblock + ch * 8), (lvoid*)&sm[buf][KCH + i * T + wave * 64], 16, 0, 0);
        }
    };
    const float scale2 = score_scale2(a.scale);
    const uint32_t vplace = (lane & 15) * 4 + ((lane >> 4) ^ value_place(lane & 15));
    if (s0 < s1) load_step(s0 & 1, s0);
    for (uint32_t s = s0; s < s1; s++) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (s + 1 < s1) load_step((s + 1) & 1, s + 1);
        const uint32_t first = (s * NB + group * NW) * 32;
        if (first > wave_last) continue;                                                  // nothing here is visible to this wave
        const uint4* ks = sm[s & 1] + group * (NW * 32 * KC);
        const uint4* vs = sm[s & 1] + KCH + group * (NW * VB) + vplace;
        const bool bound = first + 32 * NW - 1 > first_limit;
#pragma unroll
        for (int mp = 0; mp < MAPS; mp++) {                                               // (a map at a time: the registers of two halve the waves)
            lh_bf16x8 w[NW][3];
            lh_f32x4 sc[2 * NW];
#pragma unroll
            for (int t = 0; t < 2 * NW; t++) sc[t] = (lh_f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < DQ / 32; c++)
#pragma unroll
                for (int t = 0; t < 2 * NW; t++) {
                    const uint32_t key = t * 16 + (lane & 15), ch = mp * (DQ / 8) + c * 4 + (lane >> 4);
                    sc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(lh_bf16x8, ks[key * KC + (ch ^ (key & kSwizzle))]), qf[mp][c], sc[t], 0, 0, 0);
                }
            const float alpha = softmax_step<NW>(sc, st[mp], scale2, first, limit, bound, lane, w);
            if (__ballot(alpha != 1.0f)) {
#pragma unroll
                for (int d = 0; d < DV / 16; d++)
#pragma unroll
                    for (int r = 0; r < 4; r++) o[mp][d][r] *= alpha;
            }
#pragma unroll
            for (int b = 0; b < NW; b++) {
                constexpr int most = G == 2 ? 4 : 8, DB = DV / 16 < most ? DV / 16 : most;
#pragma unroll
                for (int d0 = 0; d0 < DV / 16; d0 += DB) {
                    lh_bf16x8 vf[DB];
#pragma unroll
                    for (int d = 0; d < DB; d++) vf[d] = __builtin_bit_cast(lh_bf16x8, vs[b * VB + (d0 + d) * 64]);
#pragma unroll
                    for (int z = 2; z >= 0; z--)
#pragma unroll
                        for (int d = 0; d < DB; d++) o[mp][d0 + d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[d], w[b][z], o[mp][d0 + d], 0, 0, 0);
                }
            }
        }
    }
    float l[MAPS];
#pragma unroll
    for (int mp = 0; mp < MAPS; mp++) l[mp] = lh_column_sum(st[mp].l);
    if constexpr (G == 2) {                                   // a map at a time through LDS
        static_assert(sizeof(sm) >= 4 * 64 * (DV / 16 * 16 + 8), "the sums of a group must fit the buffers");
        lh_f32x4* const sums = reinterpret_cast<lh_f32x4*>(&sm[0][0]) + (wave & 3) * (DV / 16) * 64 + lane;
        float2* const state = reinterpret_cast<float2*>(reinterpret_cast<lh_f32x4*>(&sm[0][0]) + 4 * (DV / 16) * 64) + (wave & 3) * 64 + lane;
#pragma unroll
        for (int mp = 0; mp < MAPS; mp++) {
            __syncthreads();
            if (group) {
#pragma unroll
                for (int d = 0; d < DV / 16; d++) sums[d * 64] = o[mp][d];
                *state = make_float2(st[mp].m, l[mp]);
            }
            __syncthreads();
            if (group) continue;
            const float2 other = *state;
            const float m = fmaxf(st[mp].m, other.x), base = m == -INFINITY ? 0.0f : m;
            const float f0 = __builtin_amdgcn_exp2f(st[mp].m - base), f1 = __builtin_amdgcn_exp2f(other.x - base);
#pragma unroll
            for (int d = 0; d < DV / 16; d++) {
                const lh_f32x4 y = sums[d * 64];
#pragma unroll
                for (int r = 0; r < 4; r++) o[mp][d][r] = __builtin_fmaf(f1, y[r], f0 * o[mp][d][r]);
            }
            l[mp] = __builtin_fmaf(f1, other.y, f0 * l[mp]);
            st[mp].m = m;
        }
        if (group) return;
    }
    if (a.splits == 1) { finish_row<DV, MAPS>(a, o, l, st[0].m, g, row, lane); return; }
    if (row >= packed) return;
    constexpr uint32_t kRow = DV + 4;
#pragma unroll
    for (int mp = 0; mp < MAPS; mp++) {
        float* r = a.partial + ((((size_t)(wrow >> 4) * a.kv_heads + g) * a.splits + split) * MAPS + mp) * 16 * kRow + (lane & 15) * kRow;
#pragma unroll
        for (int d = 0; d < DV / 16; d++) *reinterpret_cast<float4*>(r + d * 16 + (lane >> 4) * 4) = make_float4(o[mp][d][0], o[mp][d][1], o[mp][d][2], o[mp][d][3]);
        if (lane < 16) { r[DV] = st[mp].m; r[DV + 1] = l[mp]; }
    }
}

// grid: row tiles x kv heads x splits.  The blocks of the visible range are dealt out in contiguous runs to the 4 * splits
// waves of a (tile, kv head); where two blocks' operands fit the registers a wave loads one block ahead.
template <int DQ, int DV, int MAPS>
__global__ __launch_bounds__(256) void attention_split_kernel(const AttentionArgs a) {
    extern __shared__ __align__(16) float merge[];                          // [4 waves][MAPS][16 rows][DV + 4]: values, maximum, sum
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t split = blockIdx.x % a.splits, g = (blockIdx.x / a.splits) % a.kv_heads, tile = blockIdx.x / (a.splits * a.kv_heads);
    const uint32_t R = a.heads / a.kv_heads, packed = a.rows * R, start = *a.position;
    const uint32_t row0 = tile * 16, row_last = min(row0 + 16, packed) - 1, row = row0 + (lane & 15);
    const uint32_t last_key = min(start + row_last / R, a.capacity - 1), nb = last_key / 32 + 1;
    const uint32_t limit = min(start + row / R, last_key), first_limit = start + row0 / R;
    const uint32_t per = (nb + 4 * a.splits - 1) / (4 * a.splits), w = split * 4 + wave;
    const uint32_t b0 = min(w * per, nb), b1 = min(b0 + per, nb);

    lh_bf16x8 qf[MAPS][DQ / 32];
    load_queries<DQ, MAPS>(qf, a, g, row, lane);
    lh_f32x4 o[MAPS][DV / 16];
    RowState st[MAPS];
#pragma unroll
    for (int mp = 0; mp < MAPS; mp++) {
        st[mp] = RowState{-INFINITY, 0.0f};
#pragma unroll
        for (int d = 0; d < DV / 16; d++) o[mp][d] = (lh_f32x4){0.f, 0.f, 0.f, 0.f};
    }
    const uint16_t* K = static_cast<const uint16_t*>(a.keys) + (size_t)g * MAPS * DQ + (lane >> 4) * 8;
    const uint16_t* V = static_cast<const uint16_t*>(a.values) + (size_t)g * DV * 32;
    const size_t krow = (size_t)a.kv_heads * MAPS * DQ, vblock = (size_t)a.kv_heads * DV * 32;
    struct Block { u32x4 k[2][MAPS][DQ / 32], v[DV / 16]; };
    auto issue = [&](Block& f, uint32_t b) {
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const uint32_t p = min(b * 32 + t * 16 + (lane & 15), last_key);
#pragma unroll
            for (int mp = 0; mp < MAPS; mp++)
#pragma unroll
                for (int c = 0; c < DQ / 32; c++) f.k[t][mp][c] = *reinterpret_cast<const u32x4*>(K + p * krow + mp * DQ + c * 32);
        }
#pragma unroll
        for (int d = 0; d < DV / 16; d++) f.v[d] = *reinterpret_cast<const u32x4*>(V + b * vblock + ((d * 16 + (lane & 15)) * 4 + (lane >> 4)) * 8);
    };
    const float scale2 = score_scale2(a.scale);
    auto consume = [&](const Block& f, uint32_t b) {
        const bool bound = b * 32 + 31 > first_limit;
        lh_bf16x8 w[MAPS][1][3];
#pragma unroll
        for (int mp = 0; mp < MAPS; mp++) {
            lh_f32x4 s[2];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                s[t] = (lh_f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < DQ / 32; c++) s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(lh_bf16x8, f.k[t][mp][c]), qf[mp][c], s[t], 0, 0, 0);
            }
            const float alpha = softmax_step<1>(s, st[mp], scale2, b * 32, limit, bound, lane, w[mp]);
            if (__ballot(alpha != 1.0f)) {
#pragma unroll
                for (int d = 0; d < DV / 16; d++)
#pragma unroll
                    for (int r = 0; r < 4; r++) o[mp][d][r] *= alpha;
            }
        }
#pragma unroll
        for (int d = 0; d < DV / 16; d++)
#pragma unroll
            for (int mp = 0; mp < MAPS; mp++) {
#pragma unroll
                for (int z = 2; z >= 0; z--)
                    o[mp][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(lh_bf16x8, f.v[d]), w[mp][0][z], o[mp][d], 0, 0, 0);
            }
    };
    if constexpr (sizeof(Block) > 256) {                      // two blocks would not fit the registers
        for (uint32_t b = b0; b < b1; b++) {
            Block x;
            issue(x, b);
            consume(x, b);
        }
    } else if (b0 < b1) {
        Block x, y;
        issue(x, b0);
        for (uint32_t b = b0; b < b1; b += 2) {
            issue(y, min(b + 1, b1 - 1));
            consume(x, b);
            if (b + 1 < b1) {
                issue(x, min(b + 2, b1 - 1));
                consume(y, b + 1);
            }
        }
    }
    constexpr uint32_t kRow = DV + 4;
#pragma unroll
    for (int mp = 0; mp < MAPS; mp++) {
        const float l = lh_column_sum(st[mp].l);
        float* d0 = merge + ((wave * MAPS + mp) * 16 + (lane & 15)) * kRow;
        if (lane < 16) { d0[DV] = st[mp].m; d0[DV + 1] = l; }
#pragma unroll
        for (int d = 0; d < DV / 16; d++) *reinterpret_cast<float4*>(d0 + d * 16 + (lane >> 4) * 4) = make_float4(o[mp][d][0], o[mp][d][1], o[mp][d][2], o[mp][d][3]);
    }
    __syncthreads();
    float* rec = a.partial + (size_t)((tile * a.kv_heads + g) * a.splits + split) * MAPS * 16 * kRow;
    const uint32_t used = row_last - row0 + 1;
    for (uint32_t i = tid; i < (uint32_t)MAPS * used * DV; i += 256) {
        const uint32_t mp = i / (used * DV), rr = (i / DV) % used, d = i % DV;
        float m = -INFINITY, acc = 0.0f, l = 0.0f;
#pragma unroll
        for (int wv = 0; wv < 4; wv++) m = fmaxf(m, merge[((wv * MAPS + mp) * 16 + rr) * kRow + DV]);
        const float base = m == -INFINITY ? 0.0f : m;
#pragma unroll
        for (int wv = 0; wv < 4; wv++) {
            const float* s = merge + ((wv * MAPS + mp) * 16 + rr) * kRow;
            const float f = __builtin_amdgcn_exp2f(s[DV] - base);
            l += f * s[DV + 1];
            acc += f * s[d];
        }
        float* r = rec + (mp * 16 + rr) * kRow;
        r[d] = acc;
        if (d == 0) { r[DV] = m; r[DV + 1] = l; }
    }
}

// One row (a decoded token) over a context that one workgroup per kv head gets through: its waves take blocks of 32 keys in turn and meet in LDS, where the rows are
// finished.  Bound by the chain from the launch to the row and by the 65 GB/s or so that one CU reads, so everything that does not depend on the position is
// requested ahead of it -- the queries, and a wave's first block whether or not it is visible (it is in the cache) -- and there is no division and no second launch.
// 16 heads of 64 and 128 over 4 kv heads, two maps, recorded launches: 32 keys 5.6 us, 256 7.9, 512 10.4; in the split form with its merge 10.8, 12.2 and 12.3.  The
// leading arguments arrive in registers with the wave; the structure repeats them.
constexpr int kOneWaves = 8;
// Most blocks that the caller may ask of it, by the columns of a position that a CU reads: `values` of all maps' key and the value.  The split form takes a round of
// blocks for every four, so that it is the shorter way first where their number is a multiple of four.  (Times of this one over the split one's at 8, 11, 12, 15, 16, 19
// and 20 blocks, geometric means over up to six shapes: 192 columns 0.66, 0.68, 0.76, 0.77, 0.85, 0.86, 0.95; 256 0.68, 0.69, 0.79, 0.80, 0.90, 0.88, 0.97, up to 1.04;
// 320 0.83, 0.82, 0.99, 0.95, 1.13, 1.09, 1.30; 384 and 448 0.86, 0.86, 1.04, 1.04, 1.24, 1.15, 1.38.  The line is that of the positions a recorded step may reach.)
constexpr uint32_t one_blocks(uint32_t values) { return values <= 192 ? 20 : values <= 256 ? 19 : values <= 320 ? 15 : 11; }
constexpr bool one_fits(uint32_t values, uint32_t blocks) { return blocks <= (values > 256 && blocks % 4 == 0 ? 8 : one_blocks(values)); }
template <int DQ, int DV, int MAPS>
__global__ __launch_bounds__(64 * kOneWaves) void attention_one_kernel(const uint16_t* queries, const uint16_t* keys, const uint16_t* values, const uint32_t* position, uint32_t kv_heads,
                                                                       uint32_t R, uint32_t blocks, const AttentionArgs a) {
    extern __shared__ __align__(16) float merge[];                          // [waves][MAPS][R rows][DV + 4]: values, maximum, sum
    constexpr uint32_t kRow = DV + 4;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nwaves = kOneWaves, g = blockIdx.x, row = lane & 15;
    const uint16_t* K = keys + (size_t)g * MAPS * DQ + (lane >> 4) * 8;
    const uint16_t* V = values + (size_t)g * DV * 32 + ((lane & 15) * 4 + (lane >> 4)) * 8;
    const size_t krow = (size_t)kv_heads * MAPS * DQ, vblock = (size_t)kv_heads * DV * 32;
    struct Block { u32x4 k[2][MAPS][DQ / 32], v[DV / 16]; };
    auto issue = [&](Block& f, uint32_t b) {
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int mp = 0; mp < MAPS; mp++)
#pragma unroll
                for (int c = 0; c < DQ / 32; c++) f.k[t][mp][c] = *reinterpret_cast<const u32x4*>(K + (b * 32 + t * 16 + row) * krow + mp * DQ + c * 32);
#pragma unroll
        for (int d = 0; d < DV / 16; d++) f.v[d] = *reinterpret_cast<const u32x4*>(V + b * vblock + d * 512);
    };
    const uint32_t start = *position;
    lh_bf16x8 qf[MAPS][DQ / 32];
#pragma unroll
    for (int mp = 0; mp < MAPS; mp++)                         // as in load_queries, without its divisions (as one function the tiles get another schedule, see there)
#pragma unroll
        for (int c = 0; c < DQ / 32; c++) {
            const uint32_t k = c * 32 + (lane >> 4) * 8;
            u32x4 v = {0u, 0u, 0u, 0u};
            if (row < R && k < a.dim) {
                v = *reinterpret_cast<const u32x4*>(queries + ((size_t)(g * R + row) * MAPS + mp) * DQ + k);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    if (!(a.scale > 0.0f)) v[j] = a.scale < 0.0f ? v[j] ^ 0x80008000u : 0u;
                    if (k + 2 * j >= a.dim) v[j] = 0u;
                    else if (k + 2 * j + 1 >= a.dim) v[j] &= 0xFFFFu;
                }
            }
            qf[mp][c] = __builtin_bit_cast(lh_bf16x8, v);
        }
    Block x;
    issue(x, min(wave, blocks - 1));
    lh_f32x4 o[MAPS][DV / 16];
    RowState st[MAPS];
#pragma unroll
    for (int mp = 0; mp < MAPS; mp++) {
        st[mp] = RowState{-INFINITY, 0.0f};
#pragma unroll
        for (int d = 0; d < DV / 16; d++) o[mp][d] = (lh_f32x4){0.f, 0.f, 0.f, 0.f};
    }
    const float scale2 = score_scale2(a.scale);
    const uint32_t limit = min(start, 32 * blocks - 1), nb = limit / 32 + 1;
    for (uint32_t b = wave; b < nb; b += nwaves) {
        const bool bound = b * 32 + 31 > limit, more = b + nwaves < nb;
        lh_bf16x8 w[MAPS][1][3];
#pragma unroll
        for (int mp = 0; mp < MAPS; mp++) {
            lh_f32x4 s[2];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                s[t] = (lh_f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < DQ / 32; c++) s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(lh_bf16x8, x.k[t][mp][c]), qf[mp][c], s[t], 0, 0, 0);
            }
            const float alpha = softmax_step<1>(s, st[mp], scale2, b * 32, limit, bound, lane, w[mp]);
            if (__ballot(alpha != 1.0f)) {
#pragma unroll
                for (int d = 0; d < DV / 16; d++)
#pragma unroll
                    for (int r = 0; r < 4; r++) o[mp][d][r] *= alpha;
            }
        }
#pragma unroll
        for (int z = 2; z >= 0; z--)                          // (no product waits for the one before it)
#pragma unroll
            for (int d = 0; d < DV / 16; d++)
#pragma unroll
                for (int mp = 0; mp < MAPS; mp++) o[mp][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(lh_bf16x8, x.v[d]), w[mp][0][z], o[mp][d], 0, 0, 0);
        if (more) issue(x, b + nwaves);
    }
#pragma unroll
    for (int mp = 0; mp < MAPS; mp++) {
        const float l = lh_column_sum(st[mp].l);
        float* d0 = merge + ((wave * MAPS + mp) * R + row) * kRow;
        if (row < R) {
            if (lane < 16) { d0[DV] = st[mp].m; d0[DV + 1] = l; }
#pragma unroll
            for (int d = 0; d < DV / 16; d++) *reinterpret_cast<float4*>(d0 + d * 16 + (lane >> 4) * 4) = make_float4(o[mp][d][0], o[mp][d][1], o[mp][d][2], o[mp][d][3]);
        }
    }
    lh_lds_barrier();
    constexpr int C = (DV + 63) / 64;                         // a wave finishes a head, C columns a lane
    for (uint32_t r = wave; r < R; r += nwaves) {
        const uint32_t h = g * R + r;
        float v[C];
#pragma unroll
        for (int mp = 0; mp < MAPS; mp++) {
            const float2 ml = lane < nwaves ? *reinterpret_cast<const float2*>(merge + ((lane * MAPS + mp) * R + r) * kRow + DV) : make_float2(-INFINITY, 0.0f);
            const float sink = MAPS == 1 && a.sink ? a.sink[h] * kLog2e : -INFINITY, top = fmaxf(lh_group_max(ml.x, 64), sink);
            const float f = __builtin_amdgcn_exp2f(ml.x - top), inv = 1.0f / (lh_group_sum(f * ml.y, 64) + __builtin_amdgcn_exp2f(sink - top));
            float acc[C] = {};
#pragma unroll
            for (uint32_t w = 0; w < nwaves; w++) {
                const float fw = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f), (int)w));
                const float* s = merge + ((w * MAPS + mp) * R + r) * kRow + lane;
#pragma unroll
                for (int c = 0; c < C; c++) acc[c] += fw * (DV >= 64 || lane < DV ? s[64 * c] : 0.0f);
            }
#pragma unroll
            for (int c = 0; c < C; c++) v[c] = mp == 0 ? acc[c] * inv : v[c] - a.lambda * (acc[c] * inv);
        }
        float ss = 0.0f, f = 1.0f;
#pragma unroll
        for (int c = 0; c < C; c++) ss += 64 * c + lane < a.vdim ? v[c] * v[c] : 0.0f;
        if constexpr (MAPS == 2) f = rsqrtf(lh_group_sum(ss, 64) / (float)a.vdim + a.eps) * a.out_scale;
        if (MAPS == 1 && a.gate) f = lh_sigmoid(a.gate[h]);
#pragma unroll
        for (int c = 0; c < C; c++) if (64 * c + lane < a.vdim) static_cast<uint16_t*>(a.out)[(size_t)h * a.vdim + 64 * c + lane] = lh_f2bf(v[c] * f);
    }
}

template <int DQ, int DV, int MAPS>
int launch_mfma(lh_context* ctx, AttentionArgs& a, uint32_t max_position, const char* op, uint32_t& launches) {
    const uint32_t R = a.heads / a.kv_heads;
    const uint64_t packed = (uint64_t)a.rows * R, tiles16 = (packed + 15) / 16, cus = ctx->cu_count;
    const uint32_t max_blocks = (uint32_t)std::min<uint64_t>((uint64_t)max_position + a.rows, a.capacity) / 32 + 1;
    const size_t rec = (size_t)tiles16 * a.kv_heads * MAPS * 16 * (DV + 4) * 4;
    const uint32_t room = (uint32_t)std::min<size_t>(ctx->workspace_bytes / rec, kMaxSplits);
    auto merge = [&]() {
        launches++;
        return launch_merge<MAPS>(ctx, a, op);
    };
    a.partial = (float*)ctx->workspace;
    launches = 1;
    if (packed > 64) {
        constexpr int NB = MAPS * DQ + DV <= (MAPS == 1 ? 320 : 256) ? 2 : 1, G = MAPS == 1 ? NB : 1;
        const uint64_t groups = (packed + 63) / 64 * a.kv_heads;
        // Shares of four key steps at least up to a workgroup per CU, of eight up to two.  512 rows of 8 heads, two maps, with the merge: at
        // position 0 25 us in whole rows and 20 in two shares, at 1024 31 in three, 32 in six (a workgroup and a half per CU) and 30 in four.
        a.splits = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(std::max(std::min<uint64_t>(cus / groups, max_blocks / (4 * NB)),
                                                                               std::min<uint64_t>(2 * cus / groups, max_blocks / (8 * NB))), room));
        LH_REQUIRE(groups * a.splits < 0x7FFFFFFFull, "%s: %u rows", op, a.rows);
        // (one workgroup fits a CU where the sums of two maps take its registers: the longest first there, 2048 rows of 16 heads of 128 and 256
        // columns 188 us; in the order for two a CU 230)
        a.resident = MAPS * DV <= 256 ? (uint32_t)cus : UINT32_MAX;
        // One step of keys is all that there may be: the second group would only add its empty sums (rows of 1 to 64 keys, heads of 64 to 192: 6 % and at
        // most 8 slower; from 65 keys on two groups take as long, from 129 on less).
        const bool one = std::min<uint64_t>((uint64_t)max_position + a.rows, a.capacity) <= 32 * NB;
        if (G == 2 && one) hipLaunchKernelGGL((attention_tile_kernel<DQ, DV, MAPS, NB, 1>), dim3((uint32_t)(groups * a.splits)), dim3(256), 0, ctx->stream, a);
        else hipLaunchKernelGGL((attention_tile_kernel<DQ, DV, MAPS, NB, G>), dim3((uint32_t)(groups * a.splits)), dim3(256 * G), 0, ctx->stream, a);
        const int r = lh_check_launch(op);
        return r != LH_OK || a.splits == 1 ? r : merge();
    }
    if constexpr (MAPS * DV <= 256 && DQ + DV <= 448) {       // (what the registers hold)
        constexpr size_t per_row = (size_t)kOneWaves * MAPS * (DV + 4) * 4;
        if (a.rows == 1 && R <= 16 && one_fits(MAPS * DQ + DV, max_blocks) && R * per_row <= 160 * 1024) {
            if (R * per_row > 64 * 1024) {
                const int r = lh_raise_dynamic_lds(ctx, (const void*)attention_one_kernel<DQ, DV, MAPS>, R * per_row, op);
                if (r != LH_OK) return r;
            }
            hipLaunchKernelGGL((attention_one_kernel<DQ, DV, MAPS>), dim3(a.kv_heads), dim3(64 * kOneWaves), R * per_row, ctx->stream, (const uint16_t*)a.q,
                               (const uint16_t*)a.keys, (const uint16_t*)a.values, a.position, a.kv_heads, R, a.capacity / 32, a);
            return lh_check_launch(op);
        }
    }
    // one block per wave at least, no more workgroups than one per CU
    const uint64_t groups = tiles16 * a.kv_heads;
    LH_REQUIRE(room >= 1, "%s: %u heads of %u values exceed the workspace", op, a.heads, a.vdim);
    a.splits = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>({max_blocks / 4, (cus + groups - 1) / groups, room}));
    constexpr size_t lds = (size_t)4 * MAPS * 16 * (DV + 4) * 4;
    if (lds > 64 * 1024) {
        const int r = lh_raise_dynamic_lds(ctx, (const void*)attention_split_kernel<DQ, DV, MAPS>, lds, op);
        if (r != LH_OK) return r;
    }
    hipLaunchKernelGGL((attention_split_kernel<DQ, DV, MAPS>), dim3((uint32_t)(groups * a.splits)), dim3(256), lds, ctx->stream, a);
    const int r = lh_check_launch(op);
    return r != LH_OK ? r : merge();
}

template <int DQ, int DV>
int launch_maps(lh_context* ctx, AttentionArgs& a, uint32_t mp, const char* op, uint32_t& n) {
    if constexpr (DQ <= 128) if (a.maps == 2) return launch_mfma<DQ, DV, 2>(ctx, a, mp, op, n);
    return launch_mfma<DQ, DV, 1>(ctx, a, mp, op, n);
}
template <int DQ>
int launch_dv(lh_context* ctx, AttentionArgs& a, uint32_t mp, const char* op, uint32_t& n) {
    switch (a.dv) {
        case 32: return launch_maps<DQ, 32>(ctx, a, mp, op, n);
        case 64: return launch_maps<DQ, 64>(ctx, a, mp, op, n);
        case 128: return launch_maps<DQ, 128>(ctx, a, mp, op, n);
        default: return launch_maps<DQ, 256>(ctx, a, mp, op, n);
    }
}

// f32 queries, keys and values on the f32 matrix instructions (16 x 16 x 4): products and sums are those of FMA.  A workgroup takes 16
// packed rows of a kv head, its four waves the blocks of 32 keys in turn, straight from global memory; their results meet in LDS.
// A matrix instruction takes one value of k per lane, and which one is free as long as both operands agree: over the dimensions of a
// head lane group g has its g-th quarter of 16, over the keys of a tile its keys 4 g .. 4 g + 3, which is where S^T leaves the weights
// and what a value block keeps side by side.  (attention_plain_kernel reads keys a value at a time, every thread its own row: 333 rows
// of 8 heads with two maps over 64 dimensions, values of 128: 380 us; this form 27 us.)
constexpr uint32_t kWideMaxDim = 256;      // of a key, per map
template <int DV, int MAPS>
__global__ __launch_bounds__(256) void attention_wide_kernel(const AttentionArgs a) {
    constexpr int TD = DV / 16, kRow = DV + 4;
    extern __shared__ __align__(16) float dyn[];              // queries [MAPS][16][dq + 4], later results [4 waves][MAPS][16][DV + 4]
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, gr = lane >> 4, lr = lane & 15;
    const uint32_t g = blockIdx.x % a.kv_heads, R = a.heads / a.kv_heads, packed = a.rows * R, tiles = (packed + 15) / 16;
    const uint32_t row0 = (tiles - 1 - blockIdx.x / a.kv_heads) * 16, start = *a.position;          // the long tiles first
    const uint32_t row_last = min(row0 + 16, packed) - 1, last_key = min(start + row_last / R, a.capacity - 1);
    const uint32_t row = row0 + lr, limit = min(start + row / R, last_key), first_limit = start + row0 / R, ldq = a.dq + 4, nc = (a.dim + 15) / 16;
    for (uint32_t i = tid; i < MAPS * 16 * a.dq; i += 256) {
        const uint32_t k = i % a.dq, r = i / a.dq % 16, mp = i / a.dq / 16, pr = row0 + r, t = pr / R, h = g * R + pr - t * R;
        dyn[(mp * 16 + r) * ldq + k] = t < a.rows && k < a.dim ? static_cast<const float*>(a.q)[(((size_t)t * a.heads + h) * MAPS + mp) * a.dq + k] : 0.0f;
    }
    __syncthreads();
    lh_f32x4 o[MAPS][TD];
    float m[MAPS], l[MAPS];
#pragma unroll
    for (int mp = 0; mp < MAPS; mp++) {
        m[mp] = -INFINITY; l[mp] = 0.0f;
#pragma unroll
        for (int d = 0; d < TD; d++) o[mp][d] = (lh_f32x4){0.f, 0.f, 0.f, 0.f};
    }
    const float* K = static_cast<const float*>(a.keys) + (size_t)g * MAPS * a.dq;
    const float* V = static_cast<const float*>(a.values) + (size_t)g * DV * 32;
    const size_t krow = (size_t)a.kv_heads * MAPS * a.dq, vblock = (size_t)a.kv_heads * DV * 32;
    // DIAGONAL: not all of the 16 rows see all of the block's keys, or the cache's last ones lie behind the last row.
    auto block = [&](uint32_t b, auto diagonal) __attribute__((always_inline)) {
        constexpr bool DIAGONAL = decltype(diagonal)::value;
        float p[MAPS][8];
#pragma unroll
        for (int mp = 0; mp < MAPS; mp++) {
            lh_f32x4 s[2] = {(lh_f32x4){0.f, 0.f, 0.f, 0.f}, (lh_f32x4){0.f, 0.f, 0.f, 0.f}};
            const float* qr = dyn + (mp * 16 + lr) * ldq + gr * 4;
            const float *ka = K + min(b * 32 + lr, last_key) * krow + mp * a.dq + gr * 4, *kb = K + min(b * 32 + 16 + lr, last_key) * krow + mp * a.dq + gr * 4;
            for (uint32_t c0 = 0; c0 < nc; c0 += 4) {         // 64 dimensions at a time, all their loads ahead of the products
                lh_f32x4 x[4], y[4], q4[4];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const uint32_t c = min(c0 + u, nc - 1) * 16;
                    x[u] = *reinterpret_cast<const lh_f32x4*>(ka + c);
                    y[u] = *reinterpret_cast<const lh_f32x4*>(kb + c);
                    q4[u] = *reinterpret_cast<const lh_f32x4*>(qr + c);
                }
#pragma unroll
                for (int u = 0; u < 4; u++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const bool in = (c0 + u) * 16 + gr * 4 + j < a.dim;   // (what pads a key row may be anything)
                        s[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? x[u][j] : 0.0f, in ? q4[u][j] : 0.0f, s[0], 0, 0, 0);
                        s[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? y[u][j] : 0.0f, in ? q4[u][j] : 0.0f, s[1], 0, 0, 0);
                    }
            }
            float mx = -INFINITY;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                p[mp][i] = s[i >> 2][i & 3] * a.scale;
                if (DIAGONAL && b * 32 + (i >> 2) * 16 + gr * 4 + (i & 3) > limit) p[mp][i] = -INFINITY;
                mx = fmaxf(mx, p[mp][i]);
            }
            const float nm = fmaxf(m[mp], lh_column_max(mx)), base = nm == -INFINITY ? 0.0f : nm, alpha = expf(m[mp] - base);
            float sum = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; i++) { p[mp][i] = expf(p[mp][i] - base); sum += p[mp][i]; }
            l[mp] = l[mp] * alpha + sum;                      // this lane's keys; the four lanes of a row are added at the end
            m[mp] = nm;
#pragma unroll
            for (int d = 0; d < TD; d++)
#pragma unroll
                for (int r = 0; r < 4; r++) o[mp][d][r] *= alpha;
        }
#pragma unroll
        for (int d = 0; d < TD; d++) {
            const float* vr = V + b * vblock + (d * 16 + lr) * 32 + gr * 8;
            lh_f32x4 v[2] = {*reinterpret_cast<const lh_f32x4*>(vr), *reinterpret_cast<const lh_f32x4*>(vr + 4)};
            if constexpr (DIAGONAL) {
                bool odd = false;
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    if (b * 32 + (i >> 2) * 16 + gr * 4 + (i & 3) > last_key) v[i >> 2][i & 3] = 0.0f;    // may be anything
                    odd = odd || !(fabsf(v[i >> 2][i & 3]) < INFINITY);
                }
                if (__any(odd)) {                             // infinities and NaN must not meet the weight 0 of a row that does not see them
#pragma unroll
                    for (int mp = 0; mp < MAPS; mp++) {
                        // how many of each kind a row sees: 1 for inf, 64 for -inf, 4096 for NaN or an infinity whose weight is 0
                        lh_f32x4 seen = (lh_f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int i = 0; i < 8; i++) {
                            const float x = v[i >> 2][i & 3], w = p[mp][i], infinite = x == INFINITY ? 1.0f : x == -INFINITY ? 64.0f : 0.0f, none = x != x ? 4096.0f : 0.0f;
                            const bool sees = b * 32 + (i >> 2) * 16 + gr * 4 + (i & 3) <= limit;
                            seen = __builtin_amdgcn_mfma_f32_16x16x4f32(infinite + none, sees && w != 0.0f ? 1.0f : 0.0f, seen, 0, 0, 0);
                            seen = __builtin_amdgcn_mfma_f32_16x16x4f32(infinite + none != 0.0f ? 4096.0f : 0.0f, sees && w == 0.0f ? 1.0f : 0.0f, seen, 0, 0, 0);
                        }
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const uint32_t n = (uint32_t)seen[r];
                            if (n & 63u) o[mp][d][r] += INFINITY;
                            if (n >> 6 & 63u) o[mp][d][r] -= INFINITY;
                            if (n >> 12) o[mp][d][r] = __builtin_nanf("");
                        }
                    }
#pragma unroll
                    for (int i = 0; i < 8; i++) v[i >> 2][i & 3] = fabsf(v[i >> 2][i & 3]) < INFINITY ? v[i >> 2][i & 3] : 0.0f;
                }
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
#pragma unroll
                for (int mp = 0; mp < MAPS; mp++) {
                    o[mp][d] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[0][j], p[mp][j], o[mp][d], 0, 0, 0);
                    o[mp][d] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[1][j], p[mp][4 + j], o[mp][d], 0, 0, 0);
                }
            }
        }
    };
    uint32_t b = wave;
    for (; b * 32 + 31 <= min(first_limit, last_key); b += 4) block(b, std::false_type());
    for (; b * 32 <= last_key; b += 4) block(b, std::true_type());
    __syncthreads();
#pragma unroll
    for (int mp = 0; mp < MAPS; mp++) {
        float* d0 = dyn + ((wave * MAPS + mp) * 16 + lr) * kRow;
        const float sum = lh_column_sum(l[mp]);
        if (gr == 0) { d0[DV] = m[mp]; d0[DV + 1] = sum; }
#pragma unroll
        for (int d = 0; d < TD; d++) *reinterpret_cast<lh_f32x4*>(d0 + d * 16 + gr * 4) = o[mp][d];
    }
    __syncthreads();
    // a wave finishes four of the rows, 16 lanes a row
    const uint32_t r = wave * 4 + gr, pr = row0 + r, t = pr / R, h = g * R + pr - t * R;
    float f[MAPS][4];
#pragma unroll
    for (int mp = 0; mp < MAPS; mp++) {
        float top = -INFINITY, sum = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; w++) top = fmaxf(top, dyn[((w * MAPS + mp) * 16 + r) * kRow + DV]);
        const float sink = MAPS == 1 && a.sink && t < a.rows ? a.sink[h] : -INFINITY;
        top = fmaxf(top, sink);
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const float* d0 = dyn + ((w * MAPS + mp) * 16 + r) * kRow;
            f[mp][w] = expf(d0[DV] - top);
            sum += f[mp][w] * d0[DV + 1];
        }
        sum += expf(sink - top);
#pragma unroll
        for (int w = 0; w < 4; w++) f[mp][w] /= sum;
    }
    float v[TD], ss = 0.0f;
#pragma unroll
    for (int i = 0; i < TD; i++) {
        float x[MAPS];
#pragma unroll
        for (int mp = 0; mp < MAPS; mp++) {
            x[mp] = 0.0f;
#pragma unroll
            for (int w = 0; w < 4; w++) x[mp] += f[mp][w] * dyn[((w * MAPS + mp) * 16 + r) * kRow + i * 16 + lr];
        }
        v[i] = x[0];
        if constexpr (MAPS == 2) v[i] -= a.lambda * x[MAPS - 1];
        if (i * 16 + lr < a.vdim) ss += v[i] * v[i];
    }
    float z = 1.0f;
    if constexpr (MAPS == 2) z = rsqrtf(lh_group_sum(ss, 16) / (float)a.vdim + a.eps) * a.out_scale;
    if (t >= a.rows) return;
    if (MAPS == 1 && a.gate) z = lh_sigmoid(a.gate[(size_t)t * a.heads + h]);
    float* out = static_cast<float*>(a.out) + ((size_t)t * a.heads + h) * a.vdim;
#pragma unroll
    for (int i = 0; i < TD; i++) if (i * 16 + lr < a.vdim) out[i * 16 + lr] = v[i] * z;
}

// f32 queries, keys and values of a few rows on the vector ALU: a workgroup per row and head, its waves the blocks of 32 keys in turn.  Every load covers consecutive
// memory: sixteen lanes a key row, four dimensions each, whose products are added between lanes; eight lanes a column of the value block, four entries each, whose sums
// stay in the lanes until the end.  (With a key and a column a lane the 64 cache lines of every load bound it: 337 keys 15.5 us.)  Products and sums are FMA.
// (The matrix form fills 16 rows whether or not there are any and walks a context on four waves of one CU per kv head: 16 heads over 4 kv heads, two maps, 1 row of 337
// keys 25.7 us, 9.6 here; 16 rows of 1024 keys 66 and 17, one row of 4096 241 and 53.)
template <int DV, int MAPS>
__global__ __launch_bounds__(512) void attention_vector_kernel(const float* queries, const float* keys, const float* values, const uint32_t* position, uint32_t kv_heads, uint32_t heads,
                                                               uint32_t dq, const AttentionArgs a) {
    constexpr int WAVES = 8, NV = DV / 8;                     // loads of a value block
    __shared__ __align__(16) float ps[WAVES][MAPS][32], sums[WAVES][MAPS][DV];
    __shared__ float ms[WAVES][MAPS], ls[WAVES][MAPS], scratch[WAVES];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = lane >> 5, key = lane & 31, part = lane & 15;
    const uint32_t h = blockIdx.x % heads, t = blockIdx.x / heads, g = h / (heads / kv_heads);
    const size_t th = (size_t)t * heads + h;
    const uint32_t limit = min(*position + t, a.capacity - 1), nb = limit / 32 + 1;
    const size_t krow = (size_t)kv_heads * MAPS * dq, vblock = (size_t)kv_heads * DV * 32;
    const float *V = values + (size_t)g * DV * 32 + 4 * lane, *K = keys + (size_t)g * MAPS * dq;
    float m = -INFINITY, l = 0.0f, acc[MAPS][NV] = {};
    const uint32_t mp_of = MAPS == 2 ? half : 0u;
    for (uint32_t b = wave; b < nb; b += WAVES) {
        const bool bound = b * 32 + 31 > limit;
        lh_f32x4 v[NV];
#pragma unroll
        for (int i = 0; i < NV; i++) v[i] = *reinterpret_cast<const lh_f32x4*>(V + b * vblock + 256 * i);
        float s = 0.0f;                                       // of key `key`, map mp_of
#pragma unroll
        for (int mp = 0; mp < MAPS; mp++) {
            float sum[8] = {};                                // of key 4 i + lane / 16
            for (uint32_t c = part; c < dq / 4 + part; c += 16) {
                const uint32_t at = 4 * min(c, dq / 4 - 1);
                lh_f32x4 x[8], q4 = *reinterpret_cast<const lh_f32x4*>(queries + (th * MAPS + mp) * dq + at);
#pragma unroll
                for (int i = 0; i < 8; i++) x[i] = *reinterpret_cast<const lh_f32x4*>(K + min(b * 32 + 4 * i + (lane >> 4), limit) * krow + mp * dq + at);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const bool in = c < dq / 4 && 4 * c + j < a.dim;    // (what pads a key row may be anything)
                    q4[j] = in ? q4[j] : 0.0f;
#pragma unroll
                    for (int i = 0; i < 8; i++) sum[i] = __builtin_fmaf(in ? x[i][j] : 0.0f, q4[j], sum[i]);
                }
            }
#pragma unroll
            for (int i = 0; i < 8; i++) sum[i] = lh_group_sum(sum[i], 16);
            __builtin_amdgcn_wave_barrier();
            if (part == 0)
#pragma unroll
                for (int i = 0; i < 8; i++) ps[wave][mp][4 * i + (lane >> 4)] = sum[i];
            __builtin_amdgcn_wave_barrier();
        }
        s = ps[wave][mp_of][key] * a.scale;
        if (b * 32 + key > limit) s = -INFINITY;
        const float nm = fmaxf(m, lh_group_max(s, 32)), base = nm == -INFINITY ? 0.0f : nm, alpha = expf(m - base), p = expf(s - base);
        l = l * alpha + lh_group_sum(p, 32);
        m = nm;
        __builtin_amdgcn_wave_barrier();
        if (MAPS == 2 || half == 0) ps[wave][mp_of][lh_block_slot(key)] = p;
        __builtin_amdgcn_wave_barrier();
        const uint32_t slot = 4 * (lane & 7);                 // the lane's four entries of every column: keys 4 (slot / 8) + 16 (slot / 4 % 2) + 0 .. 3
        if (bound) {                                          // entries behind the row's last key may be anything
            const uint32_t first = b * 32 + 4 * (slot >> 3) + 16 * ((slot >> 2) & 1);
#pragma unroll
            for (int i = 0; i < NV; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) v[i][j] = first + j > limit ? 0.0f : v[i][j];
        }
#pragma unroll
        for (int mp = 0; mp < MAPS; mp++) {
            const float al = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, alpha), 32 * mp));
            const lh_f32x4 w4 = *reinterpret_cast<const lh_f32x4*>(&ps[wave][mp][slot]);
#pragma unroll
            for (int i = 0; i < NV; i++) {
                acc[mp][i] *= al;
#pragma unroll
                for (int j = 0; j < 4; j++) acc[mp][i] = __builtin_fmaf(v[i][j], w4[j], acc[mp][i]);
            }
        }
    }
    if (key == 0 && (MAPS == 2 || half == 0)) { ms[wave][mp_of] = m; ls[wave][mp_of] = l; }
#pragma unroll
    for (int mp = 0; mp < MAPS; mp++)
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const float x = lh_group_sum(acc[mp][i], 8);
            if ((lane & 7) == 0) sums[wave][mp][8 * i + (lane >> 3)] = x;
        }
    __syncthreads();
    float out = 0.0f;
    if (tid < DV) {
#pragma unroll
        for (int mp = 0; mp < MAPS; mp++) {
            const float sink = MAPS == 1 && a.sink ? a.sink[h] : -INFINITY;
            float top = sink;
#pragma unroll
            for (int w = 0; w < WAVES; w++) top = fmaxf(top, ms[w][mp]);
            float total = expf(sink - top), x = 0.0f;
#pragma unroll
            for (int w = 0; w < WAVES; w++) {
                const float f = expf(ms[w][mp] - top);
                total += f * ls[w][mp];
                x += f * sums[w][mp][tid];
            }
            x /= total;
            out = mp == 0 ? x : out - a.lambda * x;
        }
        if (tid >= a.vdim) out = 0.0f;
    }
    float z = 1.0f;
    if constexpr (MAPS == 2) z = rsqrtf(lh_block_sum(out * out, scratch) / (float)a.vdim + a.eps) * a.out_scale;
    if (MAPS == 1 && a.gate) z = lh_sigmoid(a.gate[th]);
    if (tid < a.vdim) static_cast<float*>(a.out)[th * a.vdim + tid] = out * z;
}

template <int DV, int MAPS>
int launch_wide(lh_context* ctx, const AttentionArgs& a, const char* op) {
    // Up to a workgroup a CU of the vector form, which is the faster one at every context and head measured there (16 rows of 16 heads over 4 kv heads, two maps: 32 keys
    // 13.3 us and 6.2, 337 27.0 and 9.8, 4096 242 and 49); two maps of 256 columns would not fit its registers.
    if constexpr (MAPS * DV <= 256) if ((uint64_t)a.rows * a.heads <= (uint64_t)ctx->cu_count) {
        hipLaunchKernelGGL((attention_vector_kernel<DV, MAPS>), dim3(a.rows * a.heads), dim3(512), 0, ctx->stream, (const float*)a.q, (const float*)a.keys, (const float*)a.values,
                           a.position, a.kv_heads, a.heads, a.dq, a);
        return lh_check_launch(op);
    }
    const uint64_t grid = ((uint64_t)a.rows * (a.heads / a.kv_heads) + 15) / 16 * a.kv_heads;
    LH_REQUIRE(grid < 0x7FFFFFFFull, "%s: %u rows", op, a.rows);
    const size_t lds = std::max<size_t>((size_t)MAPS * 16 * (a.dq + 4), (size_t)4 * MAPS * 16 * (DV + 4)) * 4;
    const int r = lh_raise_dynamic_lds(ctx, (const void*)attention_wide_kernel<DV, MAPS>, lds, op);
    if (r != LH_OK) return r;
    hipLaunchKernelGGL((attention_wide_kernel<DV, MAPS>), dim3((uint32_t)grid), dim3(256), lds, ctx->stream, a);
    return lh_check_launch(op);
}
template <int MAPS>
int launch_wide_dv(lh_context* ctx, const AttentionArgs& a, const char* op) {
    switch (a.dv) {
        case 32: return launch_wide<32, MAPS>(ctx, a, op);
        case 64: return launch_wide<64, MAPS>(ctx, a, op);
        case 128: return launch_wide<128, MAPS>(ctx, a, op);
        default: return launch_wide<256, MAPS>(ctx, a, op);
    }
}

}  // namespace

extern "C" {

uint32_t lh_attention_padded_dim(uint32_t dim) { return dim <= 32 ? 32u : dim <= 64 ? 64u : dim > 128 && dim <= 192 ? 192u : (dim + 127) / 128 * 128; }
uint32_t lh_attention_padded_vdim(uint32_t vdim) { return vdim <= 32 ? 32u : vdim <= 64 ? 64u : vdim <= 128 ? 128u : (vdim + 255) / 256 * 256; }

int lh_attention_rows_into(lh_batch* batch, const lh_buffer* q, const lh_buffer* keys, const lh_buffer* values, lh_buffer* output, int dtype,
                           const lh_buffer* position, uint32_t max_position, uint32_t rows, uint32_t heads, uint32_t kv_heads, uint32_t maps, uint32_t dim,
                           uint32_t vdim, uint32_t capacity, float scale, float lambda, float out_scale, float eps,
                           const lh_buffer* sink, const lh_buffer* gate) {
    const char* op = "attention_rows";
    LH_REQUIRE(batch, "%s: batch is null", op);
    LH_REQUIRE(dtype == LH_F32 || dtype == LH_BF16, "%s: dtype %d", op, dtype);
    LH_REQUIRE(maps == 1 || maps == 2, "%s: %u maps", op, maps);
    LH_REQUIRE(kv_heads > 0 && heads > 0 && heads % kv_heads == 0, "%s: heads %u is not a multiple of kv_heads %u", op, heads, kv_heads);
    LH_REQUIRE(dim > 0 && dim <= 4096 && vdim > 0 && vdim <= 1024, "%s: dim %u, vdim %u", op, dim, vdim);
    if (rows == 0) return LH_OK;
    LH_REQUIRE(capacity > 0 && capacity % 32 == 0 && (uint64_t)max_position + rows <= capacity, "%s: positions up to %llu in caches of %u", op,
               (unsigned long long)max_position + rows, capacity);
    AttentionArgs a{};
    a.dq = lh_attention_padded_dim(dim);
    a.dv = lh_attention_padded_vdim(vdim);
    const size_t es = dtype == LH_F32 ? 4 : 2;
    LH_NEED(q, (size_t)rows * heads * maps * a.dq * es, op, "q");
    LH_NEED(keys, (size_t)capacity * kv_heads * maps * a.dq * es, op, "keys");
    LH_NEED(values, (size_t)capacity * kv_heads * a.dv * es, op, "values");
    LH_NEED(output, (size_t)rows * heads * vdim * es, op, "output");
    LH_NEED(position, 4, op, "position");
    a.q = q->ptr; a.keys = keys->ptr; a.values = values->ptr; a.out = output->ptr; a.position = (const uint32_t*)position->ptr;
    a.rows = rows; a.heads = heads; a.kv_heads = kv_heads; a.maps = maps; a.dim = dim; a.vdim = vdim; a.capacity = capacity;
    a.scale = scale; a.lambda = lambda; a.out_scale = out_scale; a.eps = eps;
    LH_REQUIRE(maps == 1 || (!sink && !gate), "%s: a sink or a gate with two maps", op);
    if (sink) { LH_NEED(sink, (size_t)heads * 4, op, "sink"); a.sink = (const float*)sink->ptr; }
    if (gate) { LH_NEED(gate, (size_t)rows * heads * 4, op, "gate"); a.gate = (const float*)gate->ptr; }
    const bool aligned = (((uintptr_t)a.q | (uintptr_t)a.keys | (uintptr_t)a.values | (uintptr_t)a.out) & 15) == 0;
    uint32_t launches = 0;
    int r;
    if (dtype == LH_BF16 && aligned && a.dq <= (maps == 2 ? 128u : 256u) && a.dv <= 256) {
        if (a.dq == 32) r = launch_dv<32>(batch->ctx, a, max_position, op, launches);
        else if (a.dq == 64) r = launch_dv<64>(batch->ctx, a, max_position, op, launches);
        else if (a.dq == 128) r = launch_dv<128>(batch->ctx, a, max_position, op, launches);
        else if (a.dq == 192) r = launch_dv<192>(batch->ctx, a, max_position, op, launches);
        else r = launch_dv<256>(batch->ctx, a, max_position, op, launches);
    } else if (dtype == LH_F32 && aligned && a.dq <= kWideMaxDim && (a.dv == 32 || a.dv == 64 || a.dv == 128 || a.dv == 256)) {
        r = maps == 2 ? launch_wide_dv<2>(batch->ctx, a, op) : launch_wide_dv<1>(batch->ctx, a, op);
        launches = 1;
    } else {
        LH_REQUIRE((uint64_t)rows * heads < 0x7FFFFFFFull, "%s: %u rows", op, rows);
        const size_t lds = (size_t)maps * dim * 4;
        if (dtype == LH_F32) hipLaunchKernelGGL((attention_plain_kernel<float, float>), dim3(rows * heads), dim3(256), lds, batch->ctx->stream, a);
        else hipLaunchKernelGGL((attention_plain_kernel<uint16_t, uint16_t>), dim3(rows * heads), dim3(256), lds, batch->ctx->stream, a);
        launches = 1;
        r = lh_check_launch(op);
    }
    batch->dispatch_count += launches;
    return r;
}

}  // extern "C"
