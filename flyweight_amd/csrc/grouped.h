// The grouped product: its large tiles, and which tile a workgroup has.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// gemm_mfma_big.hip: fw_grouped_gemm on large tiles, for bfloat16 operands, the plain unit and outputs of bfloat16 (gated) or float32
__attribute__((visibility("hidden"))) bool fw_grouped_big_takes(int a_rows, int N, int K);
__attribute__((visibility("hidden"))) int fw_launch_grouped_big(const void* a, const int32_t* place_row, const void* w, bool tiled, const int32_t* expert_begin, void* out,
                                                                int gated, int places, int experts, int N, int K, bool tall, hipStream_t stream);

struct GroupedTile {
    int expert, row_tile, column_tile;      // expert < 0: none
};

// Expert e has the places begin[e] .. begin[e + 1] - 1, in tiles of `rows` (the last one not full), each times `columns` tiles of features. They are
// numbered expert by expert, within an expert column by column and within that over its tiles of places: the two or three tiles
// that read the same rows of W run side by side, and an expert's places stay in the L2 of the die that works through it. Workgroups are
// dealt to the eight dies in turn; a die takes an eighth of the tiles THERE ARE, which the device alone knows (the grid holds as many as there can
// be at most: dealt out by that number, the last dies had nothing to do. Eight rows of four of 32 experts, 252 tiles of at most
// 396, 50 a die, left two of the eight idle and a third with two). Every wave works it out for itself, in scalar
// registers: read with a shuffle the tile would count as different in every lane, and so would every address formed from it (each load to LDS then
// runs in a loop over the lanes' addresses: gated, 2,048 rows, 32 experts 173 us against 158).
__device__ __forceinline__ GroupedTile grouped_tile(const int32_t* __restrict__ begin, int experts, int rows, int columns) {
    const int lane = threadIdx.x & 63;
    auto scan = [&](int e0, int& mine) {            // tiles of places of expert e0 + lane, and of all up to it
        const int e = e0 + lane;
        mine = e < experts ? (begin[e + 1] - begin[e] + rows - 1) / rows : 0;
        int upto = mine;
#pragma unroll
        for (int offset = 1; offset < 64; offset <<= 1) {
            const int other = __shfl_up(upto, offset, 64);
            if (lane >= offset) upto += other;
        }
        return upto;
    };
    auto of_last = [](int v) { return __builtin_amdgcn_readlane(v, 63); };
    int mine, upto = scan(0, mine), total = of_last(upto);
    for (int e0 = 64; e0 < experts; e0 += 64) {
        int unused;
        total += of_last(scan(e0, unused));
    }
    total *= columns;
    const int per_die = (total + 7) / 8, of_die = blockIdx.x >> 3;
    const int logical = (blockIdx.x & 7) * per_die + of_die;
    const GroupedTile none = {-1, 0, 0};
    if (of_die >= per_die || logical >= total) return none;
    for (int e0 = 0, before = 0;;) {
        const unsigned long long holds = __ballot(logical < (before + upto) * columns);
        if (holds) {
            const int at = __ffsll((long long)holds) - 1;
            const int tiles_here = __builtin_amdgcn_readlane(mine, at);
            const int rest = logical - (before + __builtin_amdgcn_readlane(upto, at) - tiles_here) * columns;
            return {e0 + at, rest % tiles_here, rest / tiles_here};
        }
        before += of_last(upto);
        e0 += 64;
        if (e0 >= experts) return none;             // (not reached: logical < total)
        upto = scan(e0, mine);
    }
}
