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
// What bounds it: at the per-layer sizes (0.6 to 9.4 MB of weights) launch and the first memory
// round trip, so K is split over 4 or 8 waves until one block of loads per wave covers it, and
// tiles stay 16 x 16 for the most workgroups.
//
// How the operands are read: lane 16 g + r of an MFMA operand holds 16 bytes of row r at K chunk
// g, so loading operands directly puts neighbouring lanes in different rows, and the texture
// unit then takes one lane per cycle (96 KB per workgroup from L2: 3.8 us, against 2.0 us, which
// is the time of an almost empty launch, with four neighbouring lanes on 64 contiguous bytes).
// So a load takes row lane / 4, chunk lane % 4, and ds_bpermute moves the four dwords to the
// operand's lane.
#include "fc.hpp"

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

constexpr int kGemmMinWaves = 4, kGemmMaxWaves = 8;
// Steps per block.  6 instead of 3, or 16 waves for the longest rows, measured within 5 % at 768 x
// 3072, and 6 lost 7-12 % at 768 x 768.
constexpr int kGemmSteps = 3;

// kR: weight rows per workgroup (16 per MFMA operand).  kS: steps (64 bytes of a weight row: 4
// chunks) per block of loads.  The steps of a row go to the waves in contiguous runs: pk_steps = steps per wave << 8 |
// waves that take one more.  A wave without a step, rows beyond M, tokens beyond B and chunks
// beyond the row load something that exists and is dropped (rows and tokens are not stored,
// chunks enter as zeros).
template <int WT, int kR, int kS, bool kOutF32, int kEpi>
__global__ __launch_bounds__(kGemmMaxWaves * kWave) void gemm_kernel(
    const uint8_t* pk_W, const uint8_t* pk_x, const float* pk_w_scale, const void* pk_bias, int pk_M, int pk_K,
    int pk_B, int pk_col_tiles, int pk_steps, GemvArgs a) {
    using F = WFmt<WT>;
    constexpr int kCols = 16;
    constexpr int RT = kR / 16;             // operands of rows
    constexpr int kPitch = kR + 4;          // floats; keeps 16-byte stores aligned and spreads the banks
    constexpr int kXP = F::kXBytes / 16;    // 16-byte pieces of x per weight chunk
    constexpr int kIts = kR * kCols / (kGemmMinWaves * kWave);
    static_assert(kR % 16 == 0, "whole operands");
    extern __shared__ float red[];          // [waves][kCols][kPitch]
    a.B = pk_B;
    a.M = pk_M & kRowMask;
    const int K = pk_K;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int waves = blockDim.x / kWave;
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
    const int bb0 = threadIdx.x / kR, bb_step = blockDim.x / kR;
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
        float p[kGemmMaxWaves];
#pragma unroll
        for (int w = 0; w < kGemmMaxWaves; ++w)
            p[w] = w < kGemmMinWaves || w < waves ? red[(w * kCols + bb) * kPitch + mm] : 0.0f;
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

template <int WT>
const void* gemm_ptr(bool out_f32, int epi) {
    constexpr bool kAct = WFmt<WT>::kActF32;
    if (epi == kEpiAppend) return (const void*)&gemm_kernel<WT, 16, kGemmSteps, kAct, kEpiAppend>;
    if (epi == kEpiAppend8) {
        if constexpr (kAct) return nullptr;   // 8-bit caches sit behind bf16 activations
        else return (const void*)&gemm_kernel<WT, kHd, kGemmSteps, false, kEpiAppend8>;
    }
    return out_f32 ? (const void*)&gemm_kernel<WT, 16, kGemmSteps, true, kEpiNone>
                   : (const void*)&gemm_kernel<WT, 16, kGemmSteps, false, kEpiNone>;
}

}  // namespace

namespace kvattn_internal {

// Whether a call takes the matrix cores.  Measured against gemv.hip (us per call, graph of calls,
// MI355X; rows x K, tokens):
//   BF16  768 x 768    3: 3.7 / 3.0   16: 10.5 / 3.0   64: 35.9 / 3.2
//         768 x 3072   2: 4.3 / 4.9    3:  5.2 / 5.1   64: 55.2 / 5.4
//   INT8  768 x 3072   2: 3.9 / 4.3    3:  4.7 / 4.7   64: 50.1 / 5.0
//   FP32  768 x 768    3: 3.8 / 4.3    4:  4.2 / 4.3   64: 34.1 / 4.6
//         768 x 3072   6: 9.2 / 10.5   8: 11.0 / 10.5  64: 59.0 / 11.1
//         1600 x 6400  3: 27.7 / 24.6 (gemv.hip takes rows this long in blocks)
// So from 3 tokens on; FP32 weights, whose MFMA does a sixteenth of the work, from 4, and from 8
// where a row is long but still one block of gemv.hip.
bool gemm_takes(int w_dtype, int B, int M, int K) {
    const int from = w_dtype != KVATTN_KV_F32 ? 3 : (K > 1600 && K <= 4096 ? 8 : 4);
    if (B < from || M >= 8192 || K > (1 << 20)) return false;
    // Tall matrices stay with gemv.hip; so do grids beyond 2^31 threads.
    const long long groups = 8ll * ((M + 127) / 128) * ((B + 15) / 16);
    return groups * kGemmMaxWaves * kWave < (1ll << 31);
}

// The launch for arguments that launch_gemv has checked.  The waves split a row's steps alike
// whatever the epilogue, so that the QKV projection with the append in its epilogue sums as the
// plain one does, bit for bit.
int launch_gemm(GemvArgs a, int w_dtype, bool out_f32, int epi, void* stream) {
    const int wbytes = w_dtype == KVATTN_KV_F32 ? 4 : (w_dtype == KVATTN_KV_BF16 ? 2 : 1);
    constexpr int cols = 16;
    int col_tiles = (a.B + cols - 1) / cols;
    const int rows = epi == kEpiAppend8 ? kHd : 16;
    const void* fn = nullptr;
    switch (w_dtype) {
        case KVATTN_KV_F32: fn = gemm_ptr<KVATTN_KV_F32>(out_f32, epi); break;
        case KVATTN_KV_BF16: fn = gemm_ptr<KVATTN_KV_BF16>(out_f32, epi); break;
        case KVATTN_KV_INT8: fn = gemm_ptr<KVATTN_KV_INT8>(out_f32, epi); break;
        default: fn = gemm_ptr<KVATTN_KV_FP8_E4M3>(out_f32, epi); break;
    }
    if (!fn) return KVATTN_ERR_DTYPE;
    const int steps = (a.K * wbytes / 16 + 3) / 4;
    const int waves = steps <= kGemmSteps * kGemmMinWaves ? kGemmMinWaves : kGemmMaxWaves;
    int pk_steps = (steps / waves) << 8 | (steps % waves);
    const long long row_tiles = (a.M + rows - 1) / rows;
    const long long groups = 8 * ((row_tiles + 7) / 8) * col_tiles;
    int pk_m = a.M | (a.gelu ? kGeluFlag : 0);
    const size_t lds = (size_t)waves * cols * (rows + 4) * sizeof(float);
    void* params[] = {&a.W, &a.x, &a.w_scale, &a.bias, &pk_m, &a.K, &a.B, &col_tiles, &pk_steps, &a};
    const hipError_t e = hipLaunchKernel(fn, dim3((unsigned)groups), dim3(waves * kWave), params, lds,
                                         (hipStream_t)stream);
    if (e != hipSuccess) {
        set_last_hip_error((int)e);
        return KVATTN_ERR_HIP;
    }
    return KVATTN_OK;
}

}  // namespace kvattn_internal
