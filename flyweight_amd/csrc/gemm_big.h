// The product on large tiles, called by the tile (gemm_mfma_big.h has the kernel; each of the four sources below compiles one epilogue of it).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

struct BigCall {
    const void *a, *w;
    const float* bias;
    void* out;
    int out_dtype, M, N, K;
    int rows, columns;          // of a tile (a gated one: gate and up columns together)
    int each_cu;                // workgroups on a compute unit, 1 or 2
    int slices, k_each;         // K cut over workgroups (1: not); then float32 workspace [slice][tile] and a counter a tile
    float* partials;
    int* counters;
    hipStream_t stream;
    float limit = 0.0f, alpha = 0.0f, shift = 0.0f;     // of the gated unit with clamped halves
};

// whether there is such a tile: `slices` tells those with K cut from the others
__host__ __device__ inline bool fw_big_tile_exists(int mode, int rows, int columns, int each_cu, int slices) {
    if (slices > 1) return mode != 2 && each_cu == 1 && ((columns == 128 && (rows == 64 || rows == 128)) || (columns == 256 && rows == 128));
    if (each_cu == 2) return columns == 128 && (rows == 64 || rows == 128);
    if (each_cu != 1) return false;
    if (columns == 128) return rows == 64 || rows == 128 || rows == 192;
    if (columns == 192) return rows == 64 || rows == 128 || rows == 192 || rows == 256;
    if (columns == 256) return rows == 128 || rows == 192 || rows == 256;
    return columns == 320 && rows == 256;
}

// 0, or -1 with the error set
__attribute__((visibility("hidden"))) int fw_launch_big_store(const BigCall& call);
__attribute__((visibility("hidden"))) int fw_launch_big_add(const BigCall& call);
__attribute__((visibility("hidden"))) int fw_launch_big_gated(const BigCall& call);
__attribute__((visibility("hidden"))) int fw_launch_big_clamped(const BigCall& call);
