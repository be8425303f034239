// gemm.hip -- the decode step's fully connected layer for a batch of tokens on MI355X (gfx950):
// the operation of gemv.hip, out[b][m] = act(scale_m * sum_k W[m][k] x[b][k] + bias[m]), on the
// matrix cores.
//
// gemv.hip multiplies every weight on the vector units once per token, so its time grows with the
// batch (GPT-2's four BF16 projections of one layer: 14 us for one token, 214 us for 64) while the
// bytes hardly do.  Here a workgroup owns 16 RT rows x 16 NT tokens, its waves split K, and every
// 16 rows x 64 bytes of weights meet every 16 tokens in one MFMA (16x16x32 bf16, two per chunk of
// 8-bit codes, which are exact in bf16; four 16x16x4 for FP32).  Products are exact and sums FP32,
// as on the vector units.
//
// What bounds it: at the per-layer sizes (0.6 to 4.7 MB of BF16 weights) launch and the first memory
// round trip (768 x 768, 16 tokens: 3.0 us, of 2.0 for an almost empty launch; 10.5 on the vector
// units), so K is split over 8 waves (up to rows of 1536 bytes one block of loads each), and
// tiles stay 16 x 16 for the most workgroups.
//
// How the operands are read: lane 16 g + r of an MFMA operand holds 16 bytes of row r at K chunk
// g, so loading operands directly puts neighbouring lanes in different rows, and the texture
// unit then takes one lane per cycle (96 KB per workgroup from L2: 3.8 us, against 2.0 us, which
// is the time of an almost empty launch, with four neighbouring lanes on 64 contiguous bytes).
// So a load takes row lane / 4, chunk lane % 4, and ds_bpermute moves the four dwords to the
// operand's lane.
#include "fc.hpp"

#include <algorithm>
#include <type_traits>

namespace {

typedef __bf16 Bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t U32x4 __attribute__((ext_vector_type(4)));
typedef float F32x4 __attribute__((ext_vector_type(4)));

// A lane's 16-byte chunk of 8-bit codes as 16 bf16 values, two MFMA operands of 8.  Every code
// is exact in bf16: INT8 has at most 7 significant bits and a sign (-128 = -2^7), E4M3 four.
template <bool kFp8>
__device__ __forceinline__ void codes_to_bf16(U32x4 w, Bf16x8 (&o)[2]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        uint32_t p[4];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t c = w[2 * h + i];
            if constexpr (kFp8) {
                p[2 * i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(c, 1.0f, false));
                p[2 * i + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(c, 1.0f, true));
            } else {
                float f[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) f[k] = (float)(int8_t)(c >> (8 * k));
                // The high halves of two floats whose low halves are zero.
                p[2 * i] = __builtin_amdgcn_perm(__float_as_uint(f[1]), __float_as_uint(f[0]), 0x07060302u);
                p[2 * i + 1] = __builtin_amdgcn_perm(__float_as_uint(f[3]), __float_as_uint(f[2]), 0x07060302u);
            }
        }
        o[h] = __builtin_bit_cast(Bf16x8, U32x4{p[0], p[1], p[2], p[3]});
    }
}

__device__ __forceinline__ U32x4 ld16(const uint8_t* p) { return *reinterpret_cast<const U32x4*>(p); }

// The four dwords that lane src / 4 holds.
__device__ __forceinline__ U32x4 from_lane(U32x4 v, int src) {
    U32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)v[e]);
    return o;
}

// Neighbours first, then sums of neighbours.
template <typename T, int N>
__device__ __forceinline__ T tree_sum(T (&v)[N]) {
#pragma unroll
    for (int d = 1; d < N; d *= 2)
#pragma unroll
        for (int i = 0; i + d < N; i += 2 * d) v[i] += v[i + d];
    return v[0];
}

// The products of one step, 16 rows x 16 tokens: w and x hold this lane's operand chunks.
template <int WT, int kXP>
__device__ __forceinline__ F32x4 step_product(U32x4 w, const U32x4 (&x)[kXP]) {
    const F32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (WFmt<WT>::kActF32) {
        F32x4 p[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            p[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w[e]), __uint_as_float(x[0][e]), zero, 0, 0, 0);
        return tree_sum(p);
    } else if constexpr (WFmt<WT>::k8bit) {
        Bf16x8 wf[2];
        codes_to_bf16<WT == KVATTN_KV_FP8_E4M3>(w, wf);
        F32x4 p[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
            p[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h], __builtin_bit_cast(Bf16x8, x[h]), zero, 0, 0, 0);
        return p[0] + p[1];
    } else {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(Bf16x8, w), __builtin_bit_cast(Bf16x8, x[0]),
                                                       zero, 0, 0, 0);
    }
}

// Waves per workgroup, whatever K: 4 for the 12 steps of a K = 768 row of 8-bit weights cost 1 to 4 %
// of a whole decode step (INT8, 12 tokens, 4 layers: 101.0 us, 97.8 with 8).
constexpr int kGemmWaves = 8;
// Steps per block.  6 instead of 3, or 16 waves for the longest rows, measured within 5 % at 768 x
// 3072, and 6 lost 7-12 % at 768 x 768.
constexpr int kGemmSteps = 3;

// kR: weight rows per workgroup (16 per MFMA operand).  kS: steps (64 bytes of a weight row: 4
// chunks) per block of loads.  The steps of a row go to the waves in contiguous runs: pk_steps = steps per wave << 8 |
// waves that take one more.  A wave without a step, rows beyond M, tokens beyond B and chunks
// beyond the row load something that exists and is dropped (rows and tokens are not stored,
// chunks enter as zeros).
template <int WT, int kR, int kS, bool kOutF32, int kEpi>
__global__ __launch_bounds__(kGemmWaves * kWave) void gemm_kernel(
    const uint8_t* pk_W, const uint8_t* pk_x, const float* pk_w_scale, const void* pk_bias, int pk_M, int pk_K,
    int pk_B, int pk_col_tiles, int pk_steps, GemvArgs a) {
    using F = WFmt<WT>;
    constexpr int kCols = 16;
    constexpr int RT = kR / 16;             // operands of rows
    constexpr int kPitch = kR + 4;          // floats; keeps 16-byte stores aligned and spreads the banks
    constexpr int kXP = F::kXBytes / 16;    // 16-byte pieces of x per weight chunk
    constexpr int kIts = (kR * kCols + kGemmWaves * kWave - 1) / (kGemmWaves * kWave);
    static_assert(kR % 16 == 0, "whole operands");
    extern __shared__ float red[];          // [waves][kCols][kPitch]
    a.B = pk_B;
    a.M = pk_M & kRowMask;
    const int K = pk_K;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    // The column tiles of a row tile sit next to each other on one XCD (workgroups x and x + 8),
    // so that its L2 fetches the row tile's weights once.
    const int j8 = blockIdx.x >> 3;
    const int mq = div_uniform(j8, pk_col_tiles);
    const int m0 = (mq * 8 + (blockIdx.x & 7)) * kR, b0 = (j8 - mq * pk_col_tiles) * kCols;
    if (m0 >= a.M) return;   // the whole workgroup
    const int nch = K * F::kWBytes / 16;
    const int s0 = wave * (pk_steps >> 8) + min(wave, pk_steps & 255);
    const int s1 = s0 + (pk_steps >> 8) + (wave < (pk_steps & 255) ? 1 : 0);
    const int lr = lane >> 2, lc = lane & 3;   // this lane's row (or token) and chunk of a load
    const uint8_t* wp[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) wp[i] = pk_W + (size_t)min(m0 + 16 * i + lr, a.M - 1) * K * F::kWBytes;
    const uint8_t* xp = pk_x + (size_t)min(b0 + lr, a.B - 1) * K * (F::kActF32 ? 4 : 2);

    struct Block {
        U32x4 w[kS][RT];
        U32x4 x[kS][kXP];
    };
    auto load = [&](Block& t, int s) {
#pragma unroll
        for (int u = 0; u < kS; ++u) {
            const uint32_t c = (uint32_t)min((s + u) * 4 + lc, nch - 1);
#pragma unroll
            for (int i = 0; i < RT; ++i) t.w[u][i] = ld16(wp[i] + c * 16u);
#pragma unroll
            for (int h = 0; h < kXP; ++h) t.x[u][h] = ld16(xp + c * (uint32_t)F::kXBytes + 16 * h);
        }
    };
    Block t;
    load(t, s0);
    // What the epilogue needs, requested behind the first block: this thread's row is the same in
    // every round of its store loop.
    const int mm = threadIdx.x % kR, m = m0 + mm;
    const int bb0 = threadIdx.x / kR;
    constexpr int bb_step = kGemmWaves * kWave / kR;
    const int mr = min(m, a.M - 1);
    const float braw = load_act<WT>(pk_bias ? pk_bias : (const void*)pk_x, pk_bias ? mr : 0);
    const float bias = pk_bias ? braw : 0.0f;
    const float ws = F::k8bit ? pk_w_scale[mr] : 1.0f;
    int len[kIts];
    if constexpr (kEpi != kEpiNone) {
#pragma unroll
        for (int it = 0; it < kIts; ++it)
            len[it] = a.cur_len[a.lens_per_seq ? min(b0 + bb0 + it * bb_step, a.B - 1) : 0];
    }

    // FP32 sums: every step's products are summed by MFMAs that start from zero and added, on the
    // vector units, to a sum of their own for each step of a block; those are then added up as a
    // tree, and so are the waves' sums below.  The chains of roundings are then no longer than
    // gemv.hip's (48 products per lane at K = 3072, and a tree).
    F32x4 acc[RT][kS];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int u = 0; u < kS; ++u) acc[i][u] = F32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // The lane that loaded what lane 16 g + r of an operand holds: row (or token) r, chunk g.
    const int src = (((lane & 15) << 2) | (lane >> 4)) * 4;
    for (int s = s0; s < s1; s += kS) {
        if (s > s0) load(t, s);
#pragma unroll
        for (int u = 0; u < kS; ++u) {
            if (s + u >= s1) break;
            if ((s + u) * 4 + 4 > nch) {   // the row's last, partial step
                const bool live = (s + u) * 4 + lc < nch;
                const U32x4 z = {0u, 0u, 0u, 0u};
#pragma unroll
                for (int i = 0; i < RT; ++i) t.w[u][i] = live ? t.w[u][i] : z;
#pragma unroll
                for (int h = 0; h < kXP; ++h) t.x[u][h] = live ? t.x[u][h] : z;
            }
            U32x4 xs[kXP];
#pragma unroll
            for (int h = 0; h < kXP; ++h) xs[h] = from_lane(t.x[u][h], src);
#pragma unroll
            for (int i = 0; i < RT; ++i) acc[i][u] += step_product<WT>(from_lane(t.w[u][i], src), xs);
        }
    }
    // Lane 16 g + r holds rows 4 g .. 4 g + 3 of token r.
#pragma unroll
    for (int i = 0; i < RT; ++i)
        *reinterpret_cast<F32x4*>(red + (wave * kCols + (lane & 15)) * kPitch + 16 * i + 4 * (lane >> 4)) =
            tree_sum(acc[i]);
    __syncthreads();
#pragma unroll
    for (int it = 0; it < kIts; ++it) {
        const int bb = bb0 + it * bb_step, b = b0 + bb;
        if (bb >= kCols || m >= a.M || b >= a.B) continue;
        float p[kGemmWaves];
#pragma unroll
        for (int w = 0; w < kGemmWaves; ++w) p[w] = red[(w * kCols + bb) * kPitch + mm];
        float pre = tree_sum(p) * ws + bias;
        const size_t o = (size_t)b * a.M + m;
        if (a.pre_gelu) store_res<kOutF32>(a.pre_gelu, o, pre);
        if (pk_M & kGeluFlag) pre = gelu_tanh(pre);
        store_res<kOutF32>(a.out, o, pre);
        if constexpr (kEpi != kEpiNone) {
            // Output m is channel m % 64 of head h of part q/k/v; K and V rows also go to the cache.
            const int part = m / (a.NH * kHd);
            if (part == 0) continue;
            const int h = (m - part * a.NH * kHd) / kHd, c = m & (kHd - 1);
            const size_t row = cache_row_at(a, b, part, h, len[it]);
            if constexpr (kEpi == kEpiAppend) {
                store_act<WT>(a.kv, row * kHd + c, pre);
            } else {
                // A wave holds one token's head row (64 rows per workgroup, M = 3 NH 64): the
                // append's quantiser on the bf16 values that qkv holds.
                static_assert(kEpi != kEpiAppend8 || kR == kHd, "a head row per wave");
                const float x = bf16_to_f32(f32_to_bf16(pre));
                const float amax = wave_max(fabsf(x));
                const bool fp8 = a.kv_dtype == KVATTN_KV_FP8_E4M3;
                const float scale = amax / (fp8 ? kW8Limit<KVATTN_KV_FP8_E4M3> : kW8Limit<KVATTN_KV_INT8>);
                a.kv[row * kHd + c] = fp8 ? w8_code<KVATTN_KV_FP8_E4M3>(x, scale) : w8_code<KVATTN_KV_INT8>(x, scale);
                if (c == 0) a.kv_scale[row] = scale;
            }
        }
    }
}

__device__ __forceinline__ U32x4 ld16_nt(const uint8_t* p) {
    return __builtin_nontemporal_load(reinterpret_cast<const U32x4*>(p));
}

// Streamed weights: 16 rows x 128 bytes, two steps, in two loads of whole 128-byte lines (rows 0-7
// and 8-15; the wave's low half the first 64 bytes of each, its high half the others).  Swapping
// the halves between the two registers leaves each step's 16 rows x 64 bytes in one of them.
__device__ __forceinline__ void unpair(U32x4& a, U32x4& b) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const auto p = __builtin_amdgcn_permlane32_swap(a[e], b[e], false, false);
        a[e] = p[0];
        b[e] = p[1];
    }
}

// Tall matrices (a vocabulary table) for more tokens: with 16 x 16 tiles every workgroup reads its
// tokens from L2 for its 16 rows alone (50304 x 768, 64 tokens: 309 MB of tokens for 77 MB of BF16
// weights), and each further tile of tokens reads the weights again.  Here a workgroup, one per
// CU, keeps its 16 NT tokens in LDS for their whole length, in operand order (a step's 64 lanes
// side by side), and each of its waves takes whole rows, 16 at a time, with no sum across waves.
// The weights are read once, non-temporally; two blocks of kTallSteps steps are in flight per
// wave, across row tiles.  50304 x 768, 64 tokens, BF16: 22.7 us (90 MB: 4.0 TB/s; 270 us on the
// vector units).  What is left above HBM's time is filling LDS before the first product
// and the 16 waves' common start and end: a CU has 12 or 13 row tiles, so a wave has one.
// (Two row tiles per wave, 8 waves: 24.8 to 27.9 us; two smaller workgroups per CU: 28.7.)
constexpr int kTallSteps = 4;
constexpr int kTallStage = 8;    // 16-byte token loads in flight per lane while LDS is filled
constexpr int kTallWaves = 16;
constexpr int kTallRows = 20000;           // from this many rows on (gemm_plan)
constexpr int kTallGroups = 256;           // workgroups: one per CU
// A row whose steps do not fill its last block gets one more step of zero tokens, which the block's
// steps beyond the row multiply: with a real step's tokens there an infinity times their zero
// weights would be NaN (and leaving those products out by a branch spills 23 to 79 registers).
__host__ __device__ constexpr int tall_steps(int nsteps) { return nsteps + (nsteps % kTallSteps != 0 ? 1 : 0); }
constexpr long long kTallLds = 144 * 1024;   // tokens, without that step
// LDS of NT token tiles.
template <int WT> constexpr long long tall_lds(int K, int NT) {
    return ((long long)K * WFmt<WT>::kWBytes / 16 + 3) / 4 * NT * kWave * WFmt<WT>::kXBytes;
}
constexpr int kTallLdsMax = 160 * 1024;      // with it: 144 KiB and a step of at most 8 KiB

template <bool kOutF32>
__device__ __forceinline__ void store_res4(void* p, size_t i, const float (&v)[4]) {
    if constexpr (kOutF32) {
        *reinterpret_cast<F32x4*>(reinterpret_cast<float*>(p) + i) = F32x4{v[0], v[1], v[2], v[3]};
    } else {
        typedef uint32_t U32x2 __attribute__((ext_vector_type(2)));
        *reinterpret_cast<U32x2*>(reinterpret_cast<uint16_t*>(p) + i) =
            U32x2{f32_to_bf16(v[0]) | (uint32_t)f32_to_bf16(v[1]) << 16,
                  f32_to_bf16(v[2]) | (uint32_t)f32_to_bf16(v[3]) << 16};
    }
}

template <int WT, int NT, bool kOutF32>
__global__ __launch_bounds__(kTallWaves * kWave) void gemm_tall_kernel(
    const uint8_t* pk_W, const uint8_t* pk_x, const float* pk_w_scale, const void* pk_bias, int pk_M, int pk_K,
    int pk_B, int pk_col_tiles, int pk_groups, GemvArgs a) {
    using F = WFmt<WT>;
    constexpr int kT = kTallSteps, kW = kTallWaves, kRows = 16;
    constexpr int kXP = F::kXBytes / 16, kPieces = kTallStage / kXP;
    extern __shared__ U32x4 xs[];           // [steps][NT][kXP][64]
    const int M = pk_M & kRowMask, K = pk_K, B = pk_B;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int j8 = blockIdx.x >> 3;
    const int mq = div_uniform(j8, pk_col_tiles);
    const int grp = mq * 8 + (blockIdx.x & 7), b0 = (j8 - mq * pk_col_tiles) * 16 * NT;
    if (grp >= pk_groups) return;
    const int nch = K * F::kWBytes / 16;
    const int nsteps = (nch + 3) / 4, nblk = (nsteps + kT - 1) / kT;
    const int src = (((lane & 15) << 2) | (lane >> 4)) * 4;
    const int lr = lane >> 2, lc = lane & 3;
    // This workgroup's row tiles, [tile0, tile1).
    const int tiles = (M + kRows - 1) / kRows;
    const int tile0 = (int)((long long)tiles * grp / pk_groups), tile1 = (int)((long long)tiles * (grp + 1) / pk_groups);

    struct Block { U32x4 w[kT]; };
    auto load = [&](Block& t, int tile, int blk) {
        const int r0 = tile * kRows + (lr & 7);
        const uint8_t* p0 = pk_W + (size_t)min(r0, M - 1) * K * F::kWBytes;
        const uint8_t* p1 = pk_W + (size_t)min(r0 + 8, M - 1) * K * F::kWBytes;
#pragma unroll
        for (int u = 0; u < kT; u += 2) {
            const uint32_t c = (uint32_t)min((blk * kT + u) * 4 + 4 * (lane >> 5) + lc, nch - 1) * 16u;
            t.w[u] = ld16_nt(p0 + c);
            t.w[u + 1] = ld16_nt(p1 + c);
        }
    };
    Block wa, wb;
    int tile = tile0 + wave, blk = 0;       // what is consumed next
    int ltile = tile, lblk = 0;             // what is loaded next
    auto next = [&](Block& t) {
        if (ltile >= tile1) return false;
        load(t, ltile, lblk);
        if (++lblk == nblk) { lblk = 0; ltile += kW; }
        return true;
    };
    const bool busy = next(wa);
    bool more = next(wb);
    // Row scales and biases of the tile that is worked on, for the rows this lane stores.
    float ws[4], bias[4];
    auto load_rows = [&]() {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int mr = min(tile * kRows + 4 * lc + e, M - 1);
            ws[e] = F::k8bit ? pk_w_scale[mr] : 1.0f;
            bias[e] = pk_bias ? load_act<WT>(pk_bias, mr) : 0.0f;
        }
    };
    load_rows();
    // Tokens to LDS: chunk c of token t of tile j goes to step c / 4, lane 16 (c % 4) + t; zeros beyond the row.
    const int pieces = tall_steps(nsteps) * NT;
    for (int i0 = wave; i0 < pieces; i0 += kW * kPieces) {
        U32x4 v[kPieces][kXP];
#pragma unroll
        for (int k = 0; k < kPieces; ++k) {
            const int i = min(i0 + k * kW, pieces - 1), st = i / NT, j = i - st * NT;
            const uint8_t* p = pk_x + (size_t)min(b0 + 16 * j + lr, B - 1) * K * 2 +
                               (size_t)min(st * 4 + lc, nch - 1) * F::kXBytes;
#pragma unroll
            for (int h = 0; h < kXP; ++h) v[k][h] = ld16(p + 16 * h);
        }
#pragma unroll
        for (int k = 0; k < kPieces; ++k) {
            const int i = i0 + k * kW;
            if (i >= pieces) break;
#pragma unroll
            for (int h = 0; h < kXP; ++h) {
                if (i / NT * 4 + lc >= nch) v[k][h] = U32x4{0u, 0u, 0u, 0u};
                xs[(i * kXP + h) * kWave + lane] = from_lane(v[k][h], src);
            }
        }
    }
    __syncthreads();
    if (!busy) return;

    // FP32 sums: a block's four steps as a tree; blocks in turn to two sums, or to one with 8-bit
    // weights and 64 tokens, which leave no registers for two and have half as many blocks.
    constexpr int kSets = F::k8bit && NT == 4 ? 1 : 2;
    F32x4 acc[kSets][NT];
    // Four outputs of a token in one store, where they are aligned.
    const bool vec_ok = (((uintptr_t)a.out | (uintptr_t)a.pre_gelu) & (kOutF32 ? 15u : 7u)) == 0;
    auto clear = [&]() {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int k = 0; k < kSets; ++k) acc[k][j] = F32x4{0.0f, 0.0f, 0.0f, 0.0f};
    };
    clear();
    auto consume = [&](Block& t, auto which) {
        constexpr int q = decltype(which)::value % kSets;
        const int st0 = blk * kT;
#pragma unroll
        for (int u = 0; u < kT; u += 2) unpair(t.w[u], t.w[u + 1]);
        if ((st0 + kT) * 4 > nch) {
#pragma unroll
            for (int u = 0; u < kT; ++u)
                if ((st0 + u) * 4 + lc >= nch) t.w[u] = U32x4{0u, 0u, 0u, 0u};
        }
        F32x4 even[NT], pair[NT];
#pragma unroll
        for (int u = 0; u < kT; ++u) {
            const int st = min(st0 + u, nsteps);   // beyond the row: the step of zeros
            const U32x4 wv = from_lane(t.w[u], src);
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                U32x4 xv[kXP];
#pragma unroll
                for (int h = 0; h < kXP; ++h) xv[h] = xs[((st * NT + j) * kXP + h) * kWave + lane];
                const F32x4 v = step_product<WT>(wv, xv);
                if (u % 2 == 0) even[j] = v;
                else if (u == 1) pair[j] = even[j] + v;
                else acc[q][j] += pair[j] + (even[j] + v);
            }
        }
        if (++blk < nblk) return;
        // The tile is done: lane 16 g + r holds rows 4 g .. 4 g + 3 of token r.  Moved to lane 4 r + g,
        // four neighbouring lanes store 16 rows of one token.
        const int m = tile * kRows + 4 * lc, back = (lc * 16 + lr) * 4;
        const bool whole = M % 4 == 0 && m < M && vec_ok;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            F32x4 sum = acc[0][j];
            if constexpr (kSets == 2) sum += acc[1][j];
            const F32x4 v = __builtin_bit_cast(F32x4, from_lane(__builtin_bit_cast(U32x4, sum), back));
            const int b = b0 + 16 * j + lr;
            if (b >= B) continue;
            const size_t o = (size_t)b * M + m;
            float pre[4], act[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                pre[e] = v[e] * ws[e] + bias[e];
                act[e] = (pk_M & kGeluFlag) ? gelu_tanh(pre[e]) : pre[e];
            }
            if (whole) {
                if (a.pre_gelu) store_res4<kOutF32>(a.pre_gelu, o, pre);
                store_res4<kOutF32>(a.out, o, act);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (m + e >= M) break;
                    if (a.pre_gelu) store_res<kOutF32>(a.pre_gelu, o + e, pre[e]);
                    store_res<kOutF32>(a.out, o + e, act[e]);
                }
            }
        }
        clear();
        blk = 0;
        tile += kW;
        load_rows();
    };
    while (true) {
        consume(wa, std::integral_constant<int, 0>{});
        if (!more) break;
        more = next(wa);
        consume(wb, std::integral_constant<int, 1>{});
        if (!more) break;
        more = next(wb);
    }
}

template <int WT, int NT>
const void* tall_ptr(bool out_f32) {
    return out_f32 ? (const void*)&gemm_tall_kernel<WT, NT, true> : (const void*)&gemm_tall_kernel<WT, NT, false>;
}

// How a call runs on the matrix cores: rows (tall: per wave) and tokens per workgroup.
struct GemmPlan {
    const void* fn;
    int rows, cols;
    bool tall;
};

// fn == nullptr: no kernel for this call.
template <int WT>
GemmPlan gemm_plan(int B, int M, int K, bool out_f32, int epi) {
    constexpr bool kAct = WFmt<WT>::kActF32;
    if (epi == kEpiAppend8) {
        if constexpr (kAct) return {};   // 8-bit caches sit behind bf16 activations
        else return {(const void*)&gemm_kernel<WT, kHd, kGemmSteps, false, kEpiAppend8>, kHd, 16, false};
    }
    if (epi == kEpiAppend) return {(const void*)&gemm_kernel<WT, 16, kGemmSteps, kAct, kEpiAppend>, 16, 16, false};
    // Tall matrices whose tokens fit in LDS together (us per call, 16 x 16 tiles / tokens in LDS):
    //   50304 x 768   BF16  8: 18.8 / 17.4   16: 21.7 / 17.6   32: 31.9 / 19.0   64: 49.6 / 22.7
    //                 INT8                   16: 10.4 / 12.6   32: 16.2 / 14.9   64: 27.9 / 21.1
    //   24000 x 1024  BF16  32: 23.8 / 14.5  INT8  32: 13.7 / 11.8
    //   16384 x 768   BF16  32:  9.3 / 10.1  INT8  32:  7.7 /  8.6   64: 11.9 / 13.5
    // FP32 weights gain nothing (24000 x 1024, 64: 66.7 / 73.4).
    if constexpr (!kAct) {
        const int nt = B <= 16 ? 1 : (B <= 32 ? 2 : 4);
        if (M >= kTallRows && B > (WT == KVATTN_KV_BF16 ? 8 : 16) && tall_lds<WT>(K, nt) <= kTallLds) {
            if (nt == 4) return {tall_ptr<WT, 4>(out_f32), 16, 64, true};
            if (nt == 2) return {tall_ptr<WT, 2>(out_f32), 16, 32, true};
            if constexpr (WT == KVATTN_KV_BF16) return {tall_ptr<WT, 1>(out_f32), 16, 16, true};
        }
    }
    return {out_f32 ? (const void*)&gemm_kernel<WT, 16, kGemmSteps, true, kEpiNone>
                    : (const void*)&gemm_kernel<WT, 16, kGemmSteps, false, kEpiNone>, 16, 16, false};
}

}  // namespace

namespace kvattn_internal {

// Whether a call takes the matrix cores: from how many vectors on.  us per call, gemv.hip / this
// file (graph of calls, MI355X; vectors : us):
//   BF16   768 x   768   2: 3.1 / 3.0    3: 3.5 / 3.0      768 x  3072   4: 5.0 / 5.3    5: 5.5 / 5.3
//         1024 x  5120   3: 6.8 / 7.4    4: 7.8 / 7.4      256 x  8192   4: 9.1 / 10.2   5: 10.6 / 10.3
//          256 x 12288   3: 16.0 / 13.8                    512 x 32768   3: 32.3 / 38.5  4: 41.7 / 39.4
//   INT8   768 x   768   2: 2.9 / 3.0    3: 3.3 / 3.0      768 x  2048   3: 3.7 / 3.9    4: 4.1 / 3.9
//          768 x  8192   4: 8.3 / 9.2    5: 9.4 / 9.2      768 x 16384   4: 14.9 / 15.5  5: 17.5 / 15.5
//          768 x 20000   3: 23.9 / 18.1                    768 x 32768   3: 25.6 / 27.5  4: 32.7 / 27.6
//   FP8    256 x  3072   3: 3.8 / 4.1    4: 4.3 / 4.1      256 x 16384   4: 12.9 / 13.2  5: 15.5 / 13.3
//   FP32   768 x   320   4: 3.6 / 3.0    5: 4.0 / 3.0      768 x  1024   5: 4.4 / 5.3    7: 5.1 / 5.3
//         1024 x  1600   7: 6.4 / 6.6    8: 6.9 / 6.6      768 x  3072  11: 10.0 / 10.7 12: 10.6 / 10.7
//         1280 x  1024   4: 4.6 / 5.4    5: 5.0 / 5.4     1280 x  1600   4: 6.3 / 6.7    5: 6.8 / 6.6
//         3072 x   768   3: 4.9 / 4.9    4: 5.3 / 4.8     2048 x  4096   7: 16.1 / 16.6  8: 17.2 / 16.6
//         1280 x  4096   8: 15.6 / 17.1
//         1024 x  5120   3: 15.9 / 20.0  4: 19.8 / 20.0    256 x  6144   4: 18.1 / 18.9  5: 21.7 / 18.9
//          512 x  8192   5: 25.0 / 26.2  6: 29.4 / 26.7    512 x 16384   5: 47.6 / 53.6  6: 56.6 / 54.5
// The vector units' time grows with the vectors, this file's hardly does: from 3 on.  Few rows (up
// to 1024: 64 tiles here) that are long, but still one block of gemv.hip (16 KB), leave most of
// the chip idle here while that kernel keeps the weights in registers: 4 or 5.  Beyond a block
// gemv.hip reads the weights again for every vector: 3, from two blocks on 4.  FP32 weights, whose MFMA
// does a sixteenth of the work, come later throughout, and latest for few rows of up to one block.
bool gemm_takes(int w_dtype, int B, int M, int K) {
    const bool few = M <= 1024;
    int from = 3;
    if (w_dtype == KVATTN_KV_F32) {
        const bool mid = M <= 1536;
        if (K <= 768) from = few ? 6 : 4;
        else if (K <= 1024) from = few ? 6 : (mid ? 5 : 4);
        else if (K <= 1600) from = few ? 8 : (mid ? 5 : 4);
        else if (K <= 4096) from = few ? 12 : (M <= 1280 && K > 3072 ? 9 : 8);
        else if (few) from = K <= 5120 ? 4 : (K <= 6144 ? 5 : 6);
        else from = 4;
    } else if (few && K > 1600) {
        const int row = w_dtype == KVATTN_KV_BF16 ? 2 * K : K;
        if (row > 16384) from = row < 32768 ? 3 : 4;
        else if (w_dtype == KVATTN_KV_BF16) from = K > 4096 && K <= 6144 ? 4 : 5;
        else from = K <= 6144 ? 4 : 5;
    }
    if (B < from || K > (1 << 20)) return false;
    // Grids beyond 2^31 threads stay with gemv.hip.
    const long long groups = 8ll * ((M + 127) / 128) * ((B + 15) / 16);
    return groups * kGemmWaves * kWave < (1ll << 31);
}

// The launch for arguments that launch_gemv has checked.
int launch_gemm(GemvArgs a, int w_dtype, bool out_f32, int epi, void* stream) {
    const int wbytes = w_dtype == KVATTN_KV_F32 ? 4 : (w_dtype == KVATTN_KV_BF16 ? 2 : 1);
    const auto plan = [&](int e) -> GemmPlan {
        switch (w_dtype) {
            case KVATTN_KV_F32: return gemm_plan<KVATTN_KV_F32>(a.B, a.M, a.K, out_f32, e);
            case KVATTN_KV_BF16: return gemm_plan<KVATTN_KV_BF16>(a.B, a.M, a.K, out_f32, e);
            case KVATTN_KV_INT8: return gemm_plan<KVATTN_KV_INT8>(a.B, a.M, a.K, out_f32, e);
            default: return gemm_plan<KVATTN_KV_FP8_E4M3>(a.B, a.M, a.K, out_f32, e);
        }
    };
    GemmPlan p = plan(epi);
    if (!p.fn) return KVATTN_ERR_DTYPE;
    // The QKV projection with the append gives the plain projection's qkv bit for bit: the waves of
    // gemm_kernel split a row's steps alike whatever the epilogue, and where the plain call keeps
    // its tokens in LDS (other sums, and no epilogue there), the append is a launch of its own behind it.
    if (epi != kEpiNone) {
        const GemmPlan plain = plan(kEpiNone);
        if (plain.tall && (((uintptr_t)a.out | (uintptr_t)a.kv) & 15u) == 0) {
            const int st = launch_gemm(a, w_dtype, out_f32, kEpiNone, stream);
            if (st != KVATTN_OK) return st;
            return kvattn_cache_write(a.kv, a.kv_scale, a.out, a.B, a.NH, kHd, a.maxT, a.cur_len, a.lens_per_seq,
                                      a.kv_dtype, stream);
        }
    }
    const int steps = (a.K * wbytes / 16 + 3) / 4;
    int col_tiles = (a.B + p.cols - 1) / p.cols;
    int pk_m = a.M | (a.gelu ? kGeluFlag : 0);
    int groups = (a.M + p.rows - 1) / p.rows, waves, last;
    size_t lds;
    if (p.tall) {
        waves = kTallWaves;
        last = groups = std::min(groups, kTallGroups);
        lds = (size_t)tall_steps(steps) * (p.cols / 16) * kWave * (wbytes == 1 ? 32 : 16);
        if (lds > 64 * 1024) {
            const hipError_t e = hipFuncSetAttribute(p.fn, hipFuncAttributeMaxDynamicSharedMemorySize, kTallLdsMax);
            if (e != hipSuccess) {
                set_last_hip_error((int)e);
                return KVATTN_ERR_HIP;
            }
        }
    } else {
        waves = kGemmWaves;
        last = (steps / waves) << 8 | (steps % waves);
        lds = (size_t)waves * p.cols * (p.rows + 4) * sizeof(float);
    }
    void* params[] = {&a.W, &a.x, &a.w_scale, &a.bias, &pk_m, &a.K, &a.B, &col_tiles, &last, &a};
    const hipError_t e = hipLaunchKernel(p.fn, dim3(8u * (unsigned)((groups + 7) / 8) * (unsigned)col_tiles),
                                         dim3(waves * kWave), params, lds, (hipStream_t)stream);
    if (e != hipSuccess) {
        set_last_hip_error((int)e);
        return KVATTN_ERR_HIP;
    }
    return KVATTN_OK;
}

}  // namespace kvattn_internal
