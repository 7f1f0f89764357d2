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

// Every tile there is, as T(rows, columns, workgroups on a compute unit), and those that storing and adding products also have with K cut.
#define FW_BIG_WHOLE_TILES(T)                                                                                                                       \
    T(64, 128, 1) T(64, 128, 2) T(128, 128, 1) T(128, 128, 2) T(192, 128, 1) T(64, 192, 1) T(128, 192, 1) T(192, 192, 1) T(256, 192, 1) T(128, 256, 1) \
    T(192, 256, 1) T(256, 256, 1) T(256, 320, 1)
#define FW_BIG_CUT_TILES(T) T(64, 128, 1) T(128, 128, 1) T(128, 256, 1)

// whether there is such a tile: `slices` tells those with K cut from the others
__host__ __device__ inline bool fw_big_tile_exists(int mode, int rows, int columns, int each_cu, int slices) {
#define FW_IS(ROWS, COLUMNS, EACH) (rows == ROWS && columns == COLUMNS && each_cu == EACH) ||
    return slices > 1 ? mode != 2 && (FW_BIG_CUT_TILES(FW_IS) false) : (FW_BIG_WHOLE_TILES(FW_IS) false);
#undef FW_IS
}

// 0, or -1 with the error set
__attribute__((visibility("hidden"))) int fw_launch_big_store(const BigCall& call);
__attribute__((visibility("hidden"))) int fw_launch_big_add(const BigCall& call);
__attribute__((visibility("hidden"))) int fw_launch_big_gated(const BigCall& call);
__attribute__((visibility("hidden"))) int fw_launch_big_clamped(const BigCall& call);
