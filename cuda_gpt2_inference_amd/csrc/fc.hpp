// fc.hpp -- what the two kernels of the decode step's fully connected layer share (gemv.hip: one
// wave per output row; gemm.hip: matrix-core tiles for batches): the weight formats, the
// arguments of a call and the element-wise pieces of the epilogue.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "kvattn.h"
#include "lanes.hpp"

namespace kvattn_internal {
// The arguments of a fully connected call.
struct GemvArgs {
    void* out;
    void* pre_gelu;
    const uint8_t* W;
    const float* w_scale;
    const uint8_t* x;
    const void* bias;
    int B, M, K, gelu;
    // QKV projection with the KV append in its epilogue (kv != nullptr): out is qkv
    // [B][3][NH][64], and its K and V rows also go to column cur_len of the cache
    // [2][B][NH][maxT][64], in the activation type or (kv_dtype 8-bit) as codes with a row
    // scale in kv_scale [2][B][NH][maxT].  8-bit rows pass through `words` (tagged u64
    // [B][2][NH][64]), their wait bounded by `polls`.
    uint8_t* kv;
    const int* cur_len;
    int lens_per_seq, NH, maxT;
    int kv_dtype;
    float* kv_scale;
    unsigned long long* words;
    int polls;
};
}  // namespace kvattn_internal

namespace {

using kvattn_internal::GemvArgs;

template <int WT> struct WFmt;
template <> struct WFmt<KVATTN_KV_F32> {   // x, bias, out: float
    static constexpr int kWBytes = 4, kElems = 4, kXBytes = 16;
    static constexpr bool kActF32 = true, k8bit = false;
};
template <> struct WFmt<KVATTN_KV_BF16> {  // x, bias, out: bf16
    static constexpr int kWBytes = 2, kElems = 8, kXBytes = 16;
    static constexpr bool kActF32 = false, k8bit = false;
};
template <> struct WFmt<KVATTN_KV_INT8> {  // x, bias, out: bf16
    static constexpr int kWBytes = 1, kElems = 16, kXBytes = 32;
    static constexpr bool kActF32 = false, k8bit = true;
};
template <> struct WFmt<KVATTN_KV_FP8_E4M3> {
    static constexpr int kWBytes = 1, kElems = 16, kXBytes = 32;
    static constexpr bool kActF32 = false, k8bit = true;
};

template <int WT>
__device__ __forceinline__ float load_act(const void* p, size_t i) {
    if constexpr (WFmt<WT>::kActF32) return reinterpret_cast<const float*>(p)[i];
    else return bf16_to_f32(reinterpret_cast<const uint16_t*>(p)[i]);
}

template <int WT>
__device__ __forceinline__ void store_act(void* p, size_t i, float v) {
    if constexpr (WFmt<WT>::kActF32) reinterpret_cast<float*>(p)[i] = v;
    else reinterpret_cast<uint16_t*>(p)[i] = f32_to_bf16(v);
}

// out / pre_gelu element: float or bf16 (the output type may differ from the activations,
// as in the reference's float logits over bf16 activations).
template <bool kOutF32>
__device__ __forceinline__ void store_res(void* p, size_t i, float v) {
    if constexpr (kOutF32) reinterpret_cast<float*>(p)[i] = v;
    else reinterpret_cast<uint16_t*>(p)[i] = f32_to_bf16(v);
}

// GPT-2's GELU, tanh form: 0.5 v (1 + tanh(sqrt(2/pi) (v + 0.044715 v^3))).
__device__ __forceinline__ float gelu_tanh(float v) {
    const float cube = 0.044715f * v * v * v;
    return 0.5f * v * (1.0f + tanhf(0.7978845608028654f * (v + cube)));
}

constexpr int kHd = 64;   // head size of the QKV epilogue
// The epilogue of a launch (a template parameter, so that the plain GEMV carries none of it).
enum GemvEpilogue { kEpiNone = 0, kEpiAppend = 1, kEpiAppend8 = 2 };
// Bits of the preloaded M argument above the row count (M < 2^29): GELU, and the XCD-local
// layout of kEpiAppend8.
constexpr int kGeluFlag = 1 << 29, kXcdLocalFlag = 1 << 30, kRowMask = (1 << 29) - 1;

// Cache row (in units of kHd elements) of part 1 (K) or 2 (V), head h, sequence b at the
// position being appended: column cl = cur_len, clamped to [0, maxT - 1] as the append does.
__device__ __forceinline__ size_t cache_row_at(const GemvArgs& a, int b, int part, int h, int cl) {
    cl = cl < 0 ? 0 : (cl > a.maxT - 1 ? a.maxT - 1 : cl);
    size_t row = ((size_t)b * a.NH + h) * a.maxT + cl;
    if (part == 2) row += (size_t)a.B * a.NH * a.maxT;
    return row;
}

}  // namespace

namespace kvattn_internal {
// gemm.hip: whether a call takes the matrix cores, and its launch (arguments already checked).
__attribute__((visibility("hidden"))) bool gemm_takes(int w_dtype, int B, int M, int K);
__attribute__((visibility("hidden"))) int launch_gemm(GemvArgs a, int w_dtype, bool out_f32, int epi, void* stream);
void set_last_hip_error(int e);   // kvattn.hip: read back by kvattn_last_hip_error
int merge_poll_limit();           // kvattn.hip: kvattn_set_merge_poll_limit's bound
}
