// gemm_common.hpp -- what the fp8 GEMM sources share (gemm_fp8.hip,
// gemm_small.hip): operand and accumulator vector types, the output
// conversions, the bias loads and the arguments of one NT GEMM.
#pragma once

#include "df_common.hpp"

namespace dfk {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

template <typename T> struct OutCvt;
template <> struct OutCvt<float> {
    static __device__ __forceinline__ float cvt(float v) { return v; }
};
template <> struct OutCvt<uint16_t> {  // bf16 bits
    static __device__ __forceinline__ uint16_t cvt(float v) { return (uint16_t)f32_to_bf16_rne(v); }
};
template <> struct OutCvt<f16_t> {
    static __device__ __forceinline__ f16_t cvt(float v) { return f16_t{(uint16_t)f32_to_f16_rne(v)}; }
};
__device__ __forceinline__ float bias_ld(const float* b, int i) { return b[i]; }
__device__ __forceinline__ float bias_ld(const uint16_t* b, int i) { return bf16_to_f32(b[i]); }
__device__ __forceinline__ float bias_ld(const f16_t* b, int i) { return f16_to_f32(b[i].bits); }

// 4 consecutive outputs of one row: one 16-byte (fp32) or 8-byte (bf16) store
__device__ __forceinline__ void store4(float* p, const float* v) {
    *reinterpret_cast<f32x4*>(p) = f32x4{v[0], v[1], v[2], v[3]};
}
__device__ __forceinline__ void store4(uint16_t* p, const float* v) {
    *reinterpret_cast<u32x2*>(p) = u32x2{f32_to_bf16_rne(v[0]) | (f32_to_bf16_rne(v[1]) << 16),
                                        f32_to_bf16_rne(v[2]) | (f32_to_bf16_rne(v[3]) << 16)};
}
__device__ __forceinline__ void store4(f16_t* p, const float* v) {
    *reinterpret_cast<u32x2*>(p) = u32x2{f32_to_f16_rne(v[0]) | (f32_to_f16_rne(v[1]) << 16),
                                        f32_to_f16_rne(v[2]) | (f32_to_f16_rne(v[3]) << 16)};
}

struct GemmArgs {
    const uint8_t* A; int lda;
    const uint8_t* B; int ldb;
    int M, N, K;
    const float* sa; const float* sb;
    const void* bias; void* C; int ldc;
    float* ws; size_t ws_bytes;
    hipStream_t st;
};

// The rounds cost model's unit, a 128-byte K step of a 256x256 tile, in
// microseconds on a partly filled chip (one or two rounds: 1.4-2.0 measured;
// the low end, so that the persistent kernel is left only where it is slower).
constexpr double kStepUs = 1.5;

// gemm_small.hip: the kernel on 16*mt x 16*nt tiles whose `waves` waves share
// the reduction, and the best such tiling of one GEMM (cost in steps).
struct SmallPlan {
    int mt, nt, waves;
    double cost;
};
SmallPlan small_plan(int M, int N, int K, int cus);
void launch_small(const SmallPlan& p, int fmt_a, int fmt_b, int bias_dtype, int c_dtype, const GemmArgs& g);

}  // namespace dfk
