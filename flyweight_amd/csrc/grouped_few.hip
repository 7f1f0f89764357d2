// The experts' grouped product of a decode step: out[place] = a[row of place] . W[expert of place]^T where an expert has a few places, the experts' weights
// in operand tiles (16 rows x 32 columns, 1 KB in the order in which a wave loads an operand).
//
// Such a step reads the weights of the experts that its tokens chose and nothing else of size: it is bound by that stream. The tiles of 32 places in
// moe.hip stage weights through LDS, 128 bytes of 256 rows at a time by one or two workgroups on a compute unit. Here a wave by itself owns
// 16 or 32 places and 16 or 32 rows of W (gated: 16 gate and the 16 up rows of the same features) and walks all of K: every load of W is a
// contiguous kilobyte straight into operands of v_mfma_f32_16x16x32_bf16, nothing is staged and no wave meets another. Two chunks of k are in registers, the one that is
// multiplied and the one on its way. A place's sums have the order of k that the other grouped products have (the same bits), so its result does
// not depend on the step that it is in; dealing K to four waves that add up in LDS gave other bits and took as long or longer.
// Both products of 32 experts of 1,536 features over 2,048, four a row, 1 / 8 / 32 / 64 / 128 rows: tiles of 32 places 37 / 87 / 123 / 127 / 130 us, K over four
// waves 21 / 64 / 94 / 101 / 117, this 19 / 64 / 93 / 99 / 109 (8 rows: 388 MB at 6.1 TB/s).
#include "fw_common.h"
#include "fw_kernels.h"
#include "grouped.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;

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

// GATED: two row tiles of W hold gate and up of the same 16 features. PT: tiles of 16 places; RT: of 16 rows of W; STEPS of 32 k are a chunk.
template <bool GATED, int PT, int RT, int STEPS, typename TO>
__global__ __launch_bounds__(64) void grouped_few_kernel(const uint16_t* __restrict__ a, const int32_t* __restrict__ place_row, const uint16_t* __restrict__ w,
                                                        const int32_t* __restrict__ expert_begin, TO* __restrict__ out, int experts, int N, int K, int tiles_n,
                                                        const FewUnit unit) {
    static_assert(!GATED || RT == 2, "gate and up rows");
    const int lane = threadIdx.x, r16 = lane & 15, g = lane >> 4;
    const GroupedTile tile = grouped_tile(expert_begin, experts, 16 * PT, tiles_n);
    if (tile.expert < 0) return;
    const int first = expert_begin[tile.expert] + tile.row_tile * 16 * PT, end = expert_begin[tile.expert + 1];
    const int n0 = tile.column_tile * (GATED ? 16 : 16 * RT);

    const uint16_t* a_row[PT];
#pragma unroll
    for (int p = 0; p < PT; ++p) {
        const int place = first + p * 16 + r16 < end ? first + p * 16 + r16 : end - 1;       // places past the expert's last are computed and dropped
        a_row[p] = a + (size_t)(place_row ? place_row[place] : place) * K + g * 8;
    }
    const uint16_t* w_row[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        const int n = GATED ? n0 + r16 : n0 + t * 16 + r16;
        const size_t row = (size_t)tile.expert * (GATED ? 2 * N : N) + (n < N ? n : N - 1) + (GATED && t ? N : 0);     // features past the last too
        w_row[t] = w + (row >> 4) * ((size_t)(K >> 5) << 9) + (((g << 4) | (int)(row & 15)) << 3);
    }
    f32x4 acc[PT][RT];
#pragma unroll
    for (int p = 0; p < PT; ++p)
#pragma unroll
        for (int t = 0; t < RT; ++t) acc[p][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    struct Chunk {
        fw_bf16x8 w[RT][STEPS], a[PT][STEPS];
    };
    const int steps = K >> 5, whole = steps / STEPS, chunks = (steps + STEPS - 1) / STEPS;
    // (steps past the end of K ask for the first one again and are not multiplied)
    auto request = [&](Chunk& c, int at) {
#pragma unroll
        for (int j = 0; j < STEPS; ++j) {
            const int step = at * STEPS + j < steps ? at * STEPS + j : 0;
#pragma unroll
            for (int t = 0; t < RT; ++t) c.w[t][j] = fw_load_weights<true>(w_row[t] + ((size_t)step << 9));
#pragma unroll
            for (int p = 0; p < PT; ++p) c.a[p][j] = *reinterpret_cast<const fw_bf16x8*>(a_row[p] + step * 32);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](const Chunk& c, int at, auto past_the_end) {
#pragma unroll
        for (int j = 0; j < STEPS; ++j) {
            if (past_the_end(at * STEPS + j)) continue;
#pragma unroll
            for (int p = 0; p < PT; ++p)
#pragma unroll
                for (int t = 0; t < RT; ++t) acc[p][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c.w[t][j], c.a[p][j], acc[p][t], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto never = [](int) { return false; };
    auto ends = [&](int step) { return step >= steps; };
    Chunk even, odd;
    request(even, 0);
    request(odd, 1);
    int c = 0;
    for (; c + 4 <= whole; c += 2) {
        multiply(even, c, never);
        request(even, c + 2);
        multiply(odd, c + 1, never);
        request(odd, c + 3);
    }
    for (; c < chunks; c += 2) {
        multiply(even, c, ends);
        if (c + 2 < chunks) request(even, c + 2);
        multiply(odd, c + 1, ends);
        if (c + 3 < chunks) request(odd, c + 3);
    }
    fw_mfma_drain();     // the loop is left by a branch; the accumulators are read next

    // D layout: lane holds W rows 4 * (lane / 16) + r of a tile for place lane % 16
#pragma unroll
    for (int p = 0; p < PT; ++p) {
        const int place = first + p * 16 + r16;
        if (place >= end) continue;
#pragma unroll
        for (int t = 0; t < (GATED ? 1 : RT); ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int n = n0 + t * 16 + g * 4 + r;
                if (n >= N) continue;
                const float left = acc[p][t][r], right = acc[p][RT - 1][r];
                store_from_float(out, (size_t)place * N + n, !GATED ? left : unit.limit > 0.0f ? gf_clamped(left, right, unit) : gf_silu(left) * right);
            }
    }
}

template <bool GATED, int PT, int RT, int STEPS, typename TO>
static int launch(const void* a, const int32_t* place_row, const void* w, const int32_t* expert_begin, void* out, int places, int experts, int N, int K,
                  const FewUnit unit, hipStream_t stream) {
    const long long tiles_m = (long long)places / (16 * PT) + (experts < places ? experts : places);       // at most
    const int tiles_n = fw_ceil_div(N, GATED ? 16 : 16 * RT);
    FW_REQUIRE(tiles_m * tiles_n < (1ll << 30), "grouped_gemm_few: too many tiles");
    grouped_few_kernel<GATED, PT, RT, STEPS, TO><<<fw_ceil_div(tiles_m * tiles_n, 8) * 8, 64, 0, stream>>>(
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
    // Up to four places an expert a wave has twice the chunk on its way and the plain product 16 rows of W: few waves have to stream. Beyond, a wave reads a
    // for 32 rows of W. Both products of the experts above, 1 / 32 / 64 rows 18.7 / 92.8 / 102.5 us so, 20.0 / 92.4 / 98.9 with the larger tile from the start.
    const int few = place_tiles == 1 && places <= 4ll * experts;
    int status;
#define FW_FEW(GATED, PT, RT, STEPS, TO) launch<GATED, PT, RT, STEPS, TO>(a, place_row, w_tiled, expert_begin, out, places, experts, N, K, unit, s)
    if (gated) status = few ? FW_FEW(true, 1, 2, 8, bf16_t) : place_tiles == 1 ? FW_FEW(true, 1, 2, 4, bf16_t) : FW_FEW(true, 2, 2, 4, bf16_t);
    else status = few ? FW_FEW(false, 1, 1, 8, float) : place_tiles == 1 ? FW_FEW(false, 1, 2, 4, float) : FW_FEW(false, 2, 2, 4, float);
#undef FW_FEW
    if (status != 0) return status;
    FW_LAUNCH_CHECK("grouped_gemm_few");
    return 0;
}
