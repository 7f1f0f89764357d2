// The experts' grouped product of a decode step: out[place] = a[row of place] . W[expert of place]^T where an expert has a few places, the experts' weights
// in operand tiles (16 rows x 32 columns, 1 KB in the order in which a wave loads an operand).
//
// Such a step reads the weights of the experts that its tokens chose and nothing else of size: it is bound by that stream. The tiles of 32 places in
// moe.hip stage row-major weights through LDS, 128 bytes of 256 rows at a time by one or two workgroups on a compute unit. Here a workgroup owns 16 (or 32)
// places and 32 rows of W; its four waves take chunks of 128 k in turn, every load of W is a contiguous kilobyte straight into operands of
// v_mfma_f32_16x16x32_bf16, nothing is staged and nothing waited for inside the loop, and several workgroups share a compute unit, so that some
// stream while others start and end. The waves' sums meet in LDS and are added in wave order. Both products of 32 experts of 1,536 features over 2,048, four a
// row, 1 / 8 / 64 rows: 37 -> 21, 87 -> 65 (388 MB at 6.0 TB/s), 126 -> 101 us; a decode step of eight requests with three such layers 610 -> 506 us.
#include "fw_common.h"
#include "fw_kernels.h"
#include "grouped.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;

#define GF_CHUNK 128
#define GF_WAVES 4

struct FewUnit {
    float limit, alpha, shift;
};
// (the units of the other grouped products, bit for bit)
__device__ __forceinline__ float gf_silu(float g) {
    if (g >= 0.0f) return g / (1.0f + __expf(-g));
    const float e = __expf(g);
    return g * e / (1.0f + e);
}
__device__ __forceinline__ float gf_clamped(float gate, float up, const FewUnit unit) {
    const float g = fminf(gate, unit.limit), u = fminf(fmaxf(up, -unit.limit), unit.limit);
    return g / (1.0f + expf(-unit.alpha * g)) * (u + unit.shift);
}

// GATED: two row tiles of W hold gate and up of the same 16 features; else 32 features. PT: tiles of 16 places.
template <bool GATED, int PT, typename TO>
__global__ __launch_bounds__(GF_WAVES * 64) void grouped_few_kernel(const uint16_t* __restrict__ a, const int32_t* __restrict__ place_row, const uint16_t* __restrict__ w,
                                                                   const int32_t* __restrict__ expert_begin, TO* __restrict__ out, int experts, int N, int K,
                                                                   int tiles_n, const FewUnit unit) {
    __shared__ f32x4 partial[GF_WAVES][PT][2][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r16 = lane & 15, g = lane >> 4;
    const GroupedTile tile = grouped_tile(expert_begin, experts, 16 * PT, tiles_n);
    if (tile.expert < 0) return;
    const int first = expert_begin[tile.expert] + tile.row_tile * 16 * PT, end = expert_begin[tile.expert + 1];
    const int n0 = tile.column_tile * (GATED ? 16 : 32);

    const uint16_t* a_row[PT];
#pragma unroll
    for (int p = 0; p < PT; ++p) {
        const int place = first + p * 16 + r16 < end ? first + p * 16 + r16 : end - 1;       // places past the expert's last are computed and dropped
        a_row[p] = a + (size_t)(place_row ? place_row[place] : place) * K + g * 8;
    }
    const uint16_t* w_row[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int n = GATED ? n0 + r16 : n0 + t * 16 + r16;
        const size_t row = (size_t)tile.expert * (GATED ? 2 * N : N) + (n < N ? n : N - 1) + (GATED && t ? N : 0);     // features past the last too
        w_row[t] = w + (row >> 4) * ((size_t)(K >> 5) << 9) + (((g << 4) | (int)(row & 15)) << 3);
    }
    f32x4 acc[PT][2];
#pragma unroll
    for (int p = 0; p < PT; ++p)
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[p][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int k0 = wave * GF_CHUNK; k0 < K; k0 += GF_WAVES * GF_CHUNK) {
        fw_bf16x8 wf[2][4], af[PT][4];
        // every load unconditionally (past the end of K from column 0, and zero instead)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int t = 0; t < 2; ++t) wf[t][j] = fw_load_weights<true>(w_row[t] + (k0 + j * 32 < K ? (size_t)((k0 >> 5) + j) << 9 : 0));
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int p = 0; p < PT; ++p) {
                const fw_bf16x8 none = {0, 0, 0, 0, 0, 0, 0, 0};
                const fw_bf16x8 v = *reinterpret_cast<const fw_bf16x8*>(a_row[p] + (k0 + j * 32 < K ? k0 + j * 32 : 0));
                af[p][j] = k0 + j * 32 < K ? v : none;
            }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int p = 0; p < PT; ++p)
#pragma unroll
                for (int t = 0; t < 2; ++t) acc[p][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t][j], af[p][j], acc[p][t], 0, 0, 0);
    }
    fw_mfma_drain();     // the loop is left by a branch; the accumulators are read next
#pragma unroll
    for (int p = 0; p < PT; ++p)
#pragma unroll
        for (int t = 0; t < 2; ++t) partial[wave][p][t][lane] = acc[p][t];
    __syncthreads();

    // D layout: lane holds W rows 4 * (lane / 16) + r of a tile for place lane % 16
    auto total = [&](int p, int t) {
        f32x4 sum = partial[0][p][t][lane];
#pragma unroll
        for (int v = 1; v < GF_WAVES; ++v) sum += partial[v][p][t][lane];
        return sum;
    };
    for (int u = wave; u < (GATED ? PT : 2 * PT); u += GF_WAVES) {
        const int p = GATED ? u : u >> 1, t = u & 1;
        const int place = first + p * 16 + r16;
        const f32x4 left = total(p, GATED ? 0 : t), right = GATED ? total(p, 1) : f32x4{0.f, 0.f, 0.f, 0.f};
        if (place >= end) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int n = n0 + (GATED ? 0 : t * 16) + g * 4 + r;
            if (n >= N) continue;
            const float value = !GATED ? left[r] : unit.limit > 0.0f ? gf_clamped(left[r], right[r], unit) : gf_silu(left[r]) * right[r];
            store_from_float(out, (size_t)place * N + n, value);
        }
    }
}

template <bool GATED, int PT, typename TO>
static int launch(const void* a, const int32_t* place_row, const void* w, const int32_t* expert_begin, void* out, int places, int experts, int N, int K,
                  const FewUnit unit, hipStream_t stream) {
    const long long tiles_m = (long long)places / (16 * PT) + (experts < places ? experts : places);       // at most
    const int tiles_n = fw_ceil_div(N, GATED ? 16 : 32);
    FW_REQUIRE(tiles_m * tiles_n < (1ll << 30), "grouped_gemm_few: too many tiles");
    grouped_few_kernel<GATED, PT, TO><<<fw_ceil_div(tiles_m * tiles_n, 8) * 8, GF_WAVES * 64, 0, stream>>>(
        (const uint16_t*)a, place_row, (const uint16_t*)w, expert_begin, (TO*)out, experts, N, K, tiles_n, unit);
    return 0;
}

// fw_grouped_gemm's contract for bfloat16 operands, w [experts * N (gated: 2 N) rows][K] in operand tiles (K a multiple of 32), outputs of bfloat16 (gated) or float32.
extern "C" int fw_grouped_gemm_few(const void* a, const int32_t* place_row, const void* w_tiled, const int32_t* expert_begin, void* out, int gated, int places,
                                   int experts, int N, int K, int place_tiles, float glu_limit, float glu_alpha, float glu_shift, void* stream) {
    FW_REQUIRE(glu_limit >= 0.0f && (glu_limit == 0.0f || gated), "grouped_gemm_few: the experts' unit is silu or clamped, behind gate and up rows");
    FW_REQUIRE(places >= 0 && experts >= 1 && N > 0 && K > 0 && K % 32 == 0, "grouped_gemm_few: bad sizes places=%d experts=%d N=%d K=%d", places, experts, N, K);
    FW_REQUIRE((uintptr_t)a % 16 == 0 && (uintptr_t)w_tiled % 16 == 0, "grouped_gemm_few: operands must be 16-byte aligned");
    if (places == 0) return 0;
    const FewUnit unit = {glu_limit, glu_alpha, glu_shift};
    hipStream_t s = (hipStream_t)stream;
    int status;
    if (gated) status = place_tiles == 1 ? launch<true, 1, bf16_t>(a, place_row, w_tiled, expert_begin, out, places, experts, N, K, unit, s)
                                         : launch<true, 2, bf16_t>(a, place_row, w_tiled, expert_begin, out, places, experts, N, K, unit, s);
    else status = place_tiles == 1 ? launch<false, 1, float>(a, place_row, w_tiled, expert_begin, out, places, experts, N, K, unit, s)
                                   : launch<false, 2, float>(a, place_row, w_tiled, expert_begin, out, places, experts, N, K, unit, s);
    if (status != 0) return status;
    FW_LAUNCH_CHECK("grouped_gemm_few");
    return 0;
}
