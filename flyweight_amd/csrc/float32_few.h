// gemm_float32_few.hip: products of one or two float32 rows, bit for bit those of gemm_float32.hip
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// What both kernels' sums and epilogues have in common, and must for their bits to agree
#define PARTS 16                // of K, each summed by itself
enum { MF_STORE = 0, MF_ACCUMULATE = 1, MF_SWIGLU = 2 };

__device__ __forceinline__ float sigmoid_float32(float x) {
    const float e = expf(x >= 0.0f ? -x : x);
    return x >= 0.0f ? 1.0f / (1.0f + e) : e / (1.0f + e);
}

__attribute__((visibility("hidden"))) bool fw_gemm_float32_few_takes(int M, int N, int K, int mode, bool normed);
__attribute__((visibility("hidden"))) int fw_launch_float32_few(const float* a, const float* norm_weight, const int32_t* row_index, float eps, int one_centered,
                                                                const float* w, const float* bias, void* out, int out_dtype, int mode, int M, int N, int K,
                                                                hipStream_t stream);
