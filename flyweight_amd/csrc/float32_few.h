// gemm_float32_few.hip: products of one or two float32 rows, bit for bit those of gemm_float32.hip
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

__attribute__((visibility("hidden"))) bool fw_gemm_float32_few_takes(int M, int N, int K, int mode, bool normed);
__attribute__((visibility("hidden"))) int fw_launch_float32_few(const float* a, const float* norm_weight, const int32_t* row_index, float eps, int one_centered,
                                                                const float* w, const float* bias, void* out, int out_dtype, int mode, int M, int N, int K,
                                                                hipStream_t stream);
