// Tiled matrix product for long prompts and wide outputs: out[M][N] = a[M][K] . w[N][K]^T with
// 256 x 256 tiles. The 128 x 128 kernel beside this one moves 64 KB through a compute unit's
// vector memory path (64 bytes a clock) for every 1,024 clocks of MFMA work: at full MFMA rate
// the path would be busy all the time, and the kernel is bound by it at a third of the peak.
// Twice the tile edge halves the bytes per flop, in the memory path and in LDS alike:
//
//  * a workgroup of four waves computes 256 x 256; each wave a 128 x 128 quarter as 4 x 4 tiles of
//    v_mfma_f32_32x32x16_bf16, its 256 accumulators in the accumulation registers; one wave per
//    SIMD, so the overlap of loads, LDS reads and MFMAs is inside the wave;
//  * 256 x 32 slabs of both operands travel from global memory STRAIGHT into LDS
//    (buffer_load_dwordx4 .. lds: no staging registers, which the accumulators leave no room for),
//    three slabs ahead of the one being multiplied, four stages, one barrier per slab; rows are
//    not padded, their chunks are stored permuted against bank conflicts;
//  * workgroups are numbered so that each XCD works on a compact group of tiles.
//
// A product whose 256-row tiles would leave compute units idle takes tiles of 128 rows (each wave
// 64 rows): 2,048 rows by 3,072 features are 128 tiles of 256 x 192 but exactly 256 of 128 x 192.
// Such a tile moves more bytes per flop through LDS and the memory path, so it is used only where
// it fills the chip better.
//
// It serves where its tiles fill the chip (the caller compares the products' estimated times): 2,048 rows by 8,192 gated features
// are 512 tiles. Epilogues as the other products: store, add into the residual stream, SwiGLU
// (a tile holds 128 gate and the 128 up features of the same columns; a lane holds both of an
// element). The experts' grouped product of a prompt runs in the same loop, its tiles numbered as grouped.h says. The reference's prompt GEMM is a 64x64 tile of plain FMAs without tensor cores
// (native/include/flyweight_v2_native_kernels.hpp:233-311).
#include "fw_common.h"
#include "fw_kernels.h"
#include "grouped.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

#define BT 256                  // tile edge (rows: of the tall tiles)
#define BK 32                   // k per slab: an LDS row is 64 bytes, four 16-byte chunks
#define BSTAGES 4               // slabs in LDS: one is multiplied, three are on their way
#define BSLAB (BT * BK * 2)     // bytes of one operand's slab
#define BK_MOST (1 << 22)
#define BN_MOST (1 << 20)       // 256 rows of the output lie below BOUNDS
#define BOUNDS 0x80000000u
#define BGROUP_M 4
#define B_LOADS 4               // most wave-wide loads (16 rows of 64 bytes) per wave per operand per slab

enum { MB_STORE = 0, MB_ACCUMULATE = 1, MB_SWIGLU = 2 };

__device__ __forceinline__ float silu_big(float g) {
    if (g >= 0.0f) return g / (1.0f + __expf(-g));
    const float e = __expf(g);
    return g * e / (1.0f + e);
}
// The same without a branch and with the hardware reciprocal (within an ulp or two of the above:
// far below the bfloat16 the result is rounded to). exp(-g) overflows to infinity for very
// negative g, whose reciprocal is 0: the result is -0, as it should be.
__device__ __forceinline__ float silu_quick(float g) { return g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)); }
// two floats -> two bfloat16 in one word, round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
    const f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
// the value the neighbouring lane (lane ^ 1) holds
__device__ __forceinline__ float from_neighbour(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));
}

// A grouped product: places begin[e] .. begin[e + 1] - 1 are expert e's rows (row place_row[p] of a, or row p), w holds the experts' weights one
// behind the other.
struct BigGroups {
    const int32_t *place_row, *begin;
    int experts;
};

template <int TM, int TN>
struct BigTile {
    static constexpr int ROWS = 2 * TM * 32;               // rows of a tile
    static constexpr int WIDE = 2 * TN * 32;               // columns of a tile
    static constexpr int A_LOADS = ROWS / 64;              // wave-wide loads per wave for a slab of a (16 rows each)
    static constexpr int W_LOADS = WIDE / 64;              // and for a slab of w
    static constexpr int SLAB_LOADS = A_LOADS + W_LOADS;   // and for a slab of both operands
};

// K must be a multiple of BK (the loads go straight to LDS: nothing can be zeroed on the way), and at most BK_MOST (a
// lane's place in a tile's 256 rows is 32 bits, as it is in the output: N at most BN_MOST).
//
// Bound by the matrix cores at the clock that their power leaves (1.5 to 1.7 GHz in long runs): 65 % of a wave's cycles in MFMAs inside a
// prompt's step, 72 % of the gated product alone, 76 % of 8,192^3; the rest between the steps and at a tile's start and end. 2,048 x 8,192 gated x 2,048: 128.2 -> 117.5 us against reads and loads
// spread over whole steps with 64-bit addresses in vector registers; 2,048 x 6,144: 51.9 -> 49.4; 8,192^3: 1,185 -> 1,296 TFLOP/s.
// One barrier for two slabs (five stages) gave nothing more.
// TN: 32-column product tiles per wave, 4 (a 256 x 256 tile) or 3 (256 x 192: a width of 6,144
// features gives 192 tiles of 256 columns for 256 compute units, but exactly 256 tiles of 192).
// TM: 32-row product tiles per wave, 4 (256 rows a tile) or 2 (128 rows).
template <int MODE, typename TO, int TN, int TM, int STAGES, bool GROUPED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(STAGES == 3 ? 2 : 1, STAGES == 3 ? 2 : 1))) void gemm_mfma_big_kernel(
    const uint16_t* __restrict__ a, const uint16_t* __restrict__ w, const float* __restrict__ bias,
    TO* __restrict__ out, int M, int N, int K, int tiles_m, int tiles_n, int per_xcd, int up_offset, const BigGroups groups) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];      // [stage][a slab | w slab]
    constexpr int ROWS = BigTile<TM, TN>::ROWS, WIDE = BigTile<TM, TN>::WIDE;
    constexpr int A_LOADS = BigTile<TM, TN>::A_LOADS, W_LOADS = BigTile<TM, TN>::W_LOADS, SLAB_LOADS = BigTile<TM, TN>::SLAB_LOADS;
    constexpr int A_SLAB = ROWS * BK * 2, STAGE = A_SLAB + WIDE * BK * 2;       // bytes
    const int features = MODE == MB_SWIGLU ? BT / 2 : WIDE;
    static_assert(MODE != MB_SWIGLU || TN == 4, "the gated tile holds 128 gate and 128 up rows");
    int m0, n0;
    const int32_t* groups_rows = nullptr;
    if constexpr (GROUPED) {
        const GroupedTile tile = grouped_tile(groups.begin, groups.experts, ROWS, tiles_n);
        const int expert = tile.expert;
        if (expert < 0) return;
        m0 = tile.row_tile * ROWS;
        n0 = tile.column_tile * features;
        const int first = groups.begin[expert];
        M = groups.begin[expert + 1] - first;           // rows of this expert: places first .. first + M - 1
        w += (size_t)expert * (MODE == MB_SWIGLU ? 2 : 1) * N * K;
        out += (size_t)first * N;
        if (groups.place_row) groups_rows = groups.place_row + first;
        else a += (size_t)first * K;
    } else {
        const int total = tiles_m * tiles_n;
        const int logical = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
        if (logical >= total) return;
        const int width = BGROUP_M * tiles_n;
        const int group = logical / width;
        const int first_m = group * BGROUP_M;
        const int group_size = tiles_m - first_m < BGROUP_M ? tiles_m - first_m : BGROUP_M;
        m0 = (first_m + (logical % width) % group_size) * ROWS;
        n0 = (logical % width) / group_size * features;
    }

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;

    // The copy: a wave-wide load writes 1,024 contiguous bytes of LDS, lane l its 16 bytes at
    // l * 16: 16 rows of 64 bytes. Rows are not padded; instead the four chunks of a row are
    // stored permuted (chunk c of row r in slot c ^ ((r / 4) % 4)), so that the 16-byte operand
    // reads of 16 consecutive rows cover all 64 banks once (rows r, r + 4, r + 8, r + 12 would
    // otherwise share theirs). Lane l therefore ASKS for chunk (l % 4) ^ ((r / 4) % 4) of row
    // r = l / 4 of its 16 rows. Addresses are a base that the wave shares (the tile's first row; of a gated
    // product's w the first gate or up row: a wave's loads of w are all of one kind), a 32-bit
    // offset of the lane, and the slab's offset in a scalar register: a slab costs no vector arithmetic.
    const int w_part = MODE == MB_SWIGLU && wave >= 2 ? 1 : 0;
    const int w_first = MODE == MB_SWIGLU ? w_part * up_offset + n0 : n0;
    const uint16_t* a_base = GROUPED && groups_rows ? a : a + (size_t)m0 * K;
    const uint16_t* w_base = w + (size_t)w_first * K;
    uint32_t a_at[A_LOADS], w_at[B_LOADS];
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) {
        const int row = (wave * A_LOADS + i) * 16 + (lane >> 2);
        const int chunk = (lane & 3) ^ ((row >> 2) & 3);
        uint32_t from = row < M - m0 ? row : M - m0 - 1;        // rows past the end are computed and dropped
        if (GROUPED && groups_rows) from = groups_rows[m0 + (int)from];
        a_at[i] = from * (uint32_t)(2 * K) + chunk * 16;
    }
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i) {
        const int row = (wave * W_LOADS + i) * 16 + (lane >> 2);
        const int chunk = (lane & 3) ^ ((row >> 2) & 3);
        const int of_part = MODE == MB_SWIGLU ? row - w_part * (BT / 2) : row;
        w_at[i] = (uint32_t)(of_part < N - n0 ? of_part : N - n0 - 1) * (uint32_t)(2 * K) + chunk * 16;
    }
    const fw_buffer a_rows = fw_make_buffer(a_base), w_rows = fw_make_buffer(w_base);
    // loads from .. to - 1 of this wave's SLAB_LOADS for a slab
    auto request_part = [&](int slab, int from, int to) {
        unsigned char* stage = lds + (slab % STAGES) * STAGE;
        const int k0 = slab * (BK * 2);
#pragma unroll
        for (int i = 0; i < A_LOADS; ++i)
            if (i >= from && i < to) fw_buffer_to_lds(a_rows, stage + (wave * A_LOADS + i) * 1024, a_at[i], k0);
#pragma unroll
        for (int i = 0; i < W_LOADS; ++i)
            if (A_LOADS + i >= from && A_LOADS + i < to) fw_buffer_to_lds(w_rows, stage + A_SLAB + (wave * W_LOADS + i) * 1024, w_at[i], k0);
    };
    auto request = [&](int slab) { request_part(slab, 0, SLAB_LOADS); };

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    // this wave's rows of the a slab, and its rows of the w slab: for SwiGLU the columns of a wave
    // are 64 gate features (tiles 0, 1) and the 64 up features of the same columns (tiles 2, 3)
    const int a_row0 = wm * (TM * 32) + (lane & 31);
    int b_row[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j)
        b_row[j] = MODE == MB_SWIGLU ? (j >> 1) * (BT / 2) + wn * 64 + (j & 1) * 32 + (lane & 31) : wn * (TN * 32) + j * 32 + (lane & 31);
    // every row this lane reads is (lane % 32) plus a multiple of 32: one permutation for all
    const int swizzle = ((lane & 31) >> 2) & 3;
    int slot[BK / 16];
#pragma unroll
    for (int t = 0; t < BK / 16; ++t) slot[t] = ((2 * t + (lane >> 5)) ^ swizzle) * 16;

    // operand registers of one k16 step: the wave's row tiles of a and column tiles of w
    struct Operands {
        bf16x8 fa[TM], fb[TN];
    };
    auto read = [&](Operands& f, int slab, int t) {
        const unsigned char* sa = lds + (slab % STAGES) * STAGE;
        const unsigned char* sb = sa + A_SLAB;
#pragma unroll
        for (int i = 0; i < TM; ++i)
            f.fa[i] = *reinterpret_cast<const bf16x8*>(sa + (a_row0 + 32 * i) * (BK * 2) + slot[t]);
#pragma unroll
        for (int j = 0; j < TN; ++j)
            f.fb[j] = *reinterpret_cast<const bf16x8*>(sb + b_row[j] * (BK * 2) + slot[t]);
    };
    auto multiply = [&](const Operands& f, int first_row_tile, int row_tiles) {
#pragma unroll
        for (int i = first_row_tile; i < first_row_tile + row_tiles; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.fa[i], f.fb[j], acc[i][j], 0, 0, 0);
    };
    // Asks the scheduler to issue `count` times: `mfmas` MFMAs, then one instruction of `kind`
    // (0x100 LDS read, 0x020 global load). A wave issues in order and an MFMA holds the matrix
    // pipe for 32 clocks, so whatever sits between two MFMAs costs nothing.
#define FW_INTERLEAVE(count, mfmas, kind)                          \
    _Pragma("unroll") for (int u = 0; u < (count); ++u) {          \
        __builtin_amdgcn_sched_group_barrier(0x008, (mfmas), 0);   \
        __builtin_amdgcn_sched_group_barrier((kind), 1, 0);        \
    }
    // Tells the compiler that these operands are needed HERE, so that it waits for their LDS reads
    // before the next reads are issued and not, for all reads together, in front of the MFMAs.
    auto arrived = [&](const Operands& f) {
        asm volatile("" ::"v"(f.fa[0]), "v"(f.fa[1]), "v"(f.fa[TM - 2]), "v"(f.fa[TM - 1]), "v"(f.fb[0]), "v"(f.fb[1]), "v"(f.fb[2]), "v"(f.fb[TN - 1]));
    };
    // waits until at most `slabs` of this wave's requested slabs are still on their way (SLAB_LOADS loads each)
    auto wait_for_all_but = [&](int slabs) {
        if (slabs >= 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * SLAB_LOADS) : "memory");
        else if (slabs == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * SLAB_LOADS) : "memory");
        else if (slabs == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(1 * SLAB_LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };

    // Four stages: while slab s is multiplied, slabs s + 1 .. s + 3 are in LDS or on their way.
    // The two k16 steps of a slab are software-pipelined by hand, because with one wave per SIMD
    // nothing else hides the latency of LDS: the operands of the next step are read behind the first
    // MFMAs of this one, a read each, so that they have arrived when the step is through. Between
    // the two steps the wave makes sure that slab s + 1 has landed (its own loads: vmcnt;
    // everybody's: the barrier), which also tells that every wave has read the last of slab s,
    // whose stage then takes slab s + 4. Its loads are issued behind every second one of the later MFMAs, half
    // of them in the next slab's step 0: a compute unit takes a wave's load in 16 clocks, and four
    // waves that each issued one behind every MFMA (32 clocks) stood still at them.
    const int steps = K / BK;
    for (int s = 0; s < STAGES && s < steps; ++s) request(s);
    wait_for_all_but((steps < STAGES ? steps : STAGES) - 1);
    __builtin_amdgcn_s_barrier();
    Operands f0, f1;
    read(f0, 0, 0);
    int s = 0;
    constexpr int EARLY = SLAB_LOADS / 2;
    // (where the reads outnumber the MFMAs the rest is left to the scheduler)
#define FW_STEP_SCHEDULE()                                                                   \
    FW_INTERLEAVE((TM + TN < TM * TN ? TM + TN : TM * TN), 1, 0x100)                          \
    FW_INTERLEAVE((TM + TN < TM * TN ? (TM * TN - TM - TN) / 2 : 0), 2, 0x020)                \
    __builtin_amdgcn_sched_barrier(0);
    if (s + STAGES < steps) {
        read(f1, 0, 1);
        multiply(f0, 0, TM);
        FW_INTERLEAVE((TM + TN < TM * TN ? TM + TN : TM * TN), 1, 0x100)
        __builtin_amdgcn_sched_barrier(0);
        // a turn: step 1 of slab s and step 0 of slab s + 1, with the loads of slab s + STAGES. Nothing in it is
        // conditional, so that each step is one run of instructions the scheduler can interleave
        do {
            arrived(f1);                                    // slab s has been read
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 2) * SLAB_LOADS) : "memory");   // slab s + 1 has landed; those behind it may still fly
            __builtin_amdgcn_s_barrier();
            read(f0, s + 1, 0);
            request_part(s + STAGES, 0, EARLY);
            multiply(f1, 0, TM);
            FW_STEP_SCHEDULE()
            read(f1, s + 1, 1);
            request_part(s + STAGES, EARLY, SLAB_LOADS);
            multiply(f0, 0, TM);
            FW_STEP_SCHEDULE()
            ++s;
        } while (s + STAGES < steps);
        // step 1 of slab s = steps - STAGES, of which step 0 is done
        arrived(f1);
        wait_for_all_but(STAGES - 2);
        __builtin_amdgcn_s_barrier();
        read(f0, s + 1, 0);
        multiply(f1, 0, TM);
        __builtin_amdgcn_sched_barrier(0);
        ++s;
    }
#undef FW_STEP_SCHEDULE
    // the last slabs: nothing more to request
    for (; s < steps; ++s) {
        arrived(f0);
        read(f1, s, 1);
        multiply(f0, 0, TM);
        __builtin_amdgcn_sched_barrier(0);
        arrived(f1);
        if (s + 1 < steps) {
            wait_for_all_but(steps - 2 - s);                // slabs s + 2 .. may still fly
            __builtin_amdgcn_s_barrier();
            read(f0, s + 1, 0);
        }
        multiply(f1, 0, TM);
        __builtin_amdgcn_sched_barrier(0);
    }
#undef FW_INTERLEAVE
    fw_mfma_drain();     // branches follow that lead to code reading the accumulators

    // D layout of the 32x32 product: lane holds column lane % 32; register r is row
    // 8 * (r / 4) + 4 * (lane / 32) + r % 4
    const int col = lane & 31, row_base = (lane >> 5) * 4;
    // The output leaves through a buffer that ends behind the tile's last row, so that rows past the end are dropped by its
    // bounds and a lane of a column past the end by a place beyond them: no branch. (With a branch an element the last tile
    // of a ragged product took 5 us longer than a whole one, with one only a row 4 us: 192 x 1,536 gated x 1,024 28.7 us
    // against 22.1 for 256 rows.) For bfloat16 two neighbouring lanes swap one value each so that each stores a pair of
    // columns as one word, which takes an even N and an output at a multiple of four bytes. With one workgroup per compute
    // unit nothing runs beside the epilogue, so its length counts.
    constexpr int SIZE = sizeof(TO) == 4 ? 4 : 2;
    const int rows_here = M - m0 < ROWS ? M - m0 : ROWS;
    const fw_buffer to = fw_make_buffer(out + (size_t)m0 * N + n0, (uint32_t)(rows_here * N - n0) * SIZE);
    const uint32_t row_step = (uint32_t)N * SIZE;
    const bool odd = lane & 1;
    // (the grouped product has the unit of its form for few places, bit for bit)
    auto unit = [](float g) { return GROUPED ? silu_big(g) : silu_quick(g); };
    const uint32_t first_row = (uint32_t)(wm * (TM * 32) + row_base);      // of this lane, of the tile
    if (SIZE == 4 || ((N & 1) == 0 && (uintptr_t)out % 4 == 0)) {
#pragma unroll
        for (int j = 0; j < (MODE == MB_SWIGLU ? 2 : TN); ++j) {
            const int c = (MODE == MB_SWIGLU ? wn * 64 : wn * (TN * 32)) + j * 32 + col;        // column of the tile
            const bool there = n0 + c < N;
            if constexpr (SIZE == 4) {
                const float b = bias && there ? bias[n0 + c] : 0.0f;
                const uint32_t at = there ? first_row * row_step + c * 4 : BOUNDS;
                float old[MODE == MB_ACCUMULATE ? TM * 16 : 1];
                if constexpr (MODE == MB_ACCUMULATE) {
#pragma unroll
                    for (int u = 0; u < TM * 16; ++u)
                        old[u] = fw_buffer_load_float(to, at + (uint32_t)((u >> 4) * 32 + 8 * ((u & 15) >> 2) + (u & 3)) * row_step);
                }
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        float value = acc[i][j][r] + b;
                        if (MODE == MB_ACCUMULATE) value += old[i * 16 + r];
                        fw_buffer_store(to, at + (uint32_t)(i * 32 + 8 * (r >> 2) + (r & 3)) * row_step, __builtin_bit_cast(uint32_t, value));
                    }
            } else {
                const float b = MODE != MB_SWIGLU && bias && there ? bias[n0 + c] : 0.0f;
                const uint32_t at = there ? (first_row + (odd ? 1 : 0)) * row_step + (c & ~1) * 2 : BOUNDS;
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            const int r = 4 * q + 2 * h;        // rows 8 q + 2 h and the one below, of row tile i
                            float upper, lower;
                            if constexpr (MODE == MB_SWIGLU) {
                                upper = fw_gate_of<TO>(acc[i][j][r], unit) * acc[i][j + 2][r];
                                lower = fw_gate_of<TO>(acc[i][j][r + 1], unit) * acc[i][j + 2][r + 1];
                            } else {
                                upper = fw_before_store<TO>(acc[i][j][r] + b);
                                lower = fw_before_store<TO>(acc[i][j][r + 1] + b);
                            }
                            const float got = from_neighbour(odd ? upper : lower);
                            const uint32_t word = odd ? pack_bf16x2(got, lower) : pack_bf16x2(upper, got);
                            fw_buffer_store(to, at + (uint32_t)(i * 32 + 8 * q + 2 * h) * row_step, word);
                        }
            }
        }
        return;
    }
    // Two bytes an element, and rows of an odd length or an output at an odd place: every element leaves by itself, just as free of branches
    // (with two an element 5,532 x 83 x 608 took 19.0 us against 11.5, 1,300 x 3,071 x 1,024 25.7 against 18.3).
    if constexpr (SIZE == 2) {
#pragma unroll
        for (int j = 0; j < (MODE == MB_SWIGLU ? 2 : TN); ++j) {
            const int c = (MODE == MB_SWIGLU ? wn * 64 : wn * (TN * 32)) + j * 32 + col;
            const bool there = n0 + c < N;
            const float b = MODE != MB_SWIGLU && bias && there ? bias[n0 + c] : 0.0f;
            const uint32_t at = there ? first_row * row_step + c * 2 : BOUNDS;
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    float value;
                    if constexpr (MODE == MB_SWIGLU) value = fw_gate_of<TO>(acc[i][j][r], unit) * acc[i][j + 2][r];
                    else value = fw_before_store<TO>(acc[i][j][r] + b);
                    fw_buffer_store(to, at + (uint32_t)(i * 32 + 8 * (r >> 2) + (r & 3)) * row_step, float_to_bf16_bits(value));
                }
        }
    }
}

template <int MODE, typename TO, int TN, int TM, int STAGES, bool GROUPED>
static int launch_tiles(const void* a, const void* w, const float* bias, void* out, int M, int N, int K, int tiles_m, const BigGroups& groups,
                        hipStream_t stream) {
    const int tiles_n = fw_ceil_div(N, MODE == MB_SWIGLU ? BT / 2 : BigTile<TM, TN>::WIDE);
    const int per_xcd = fw_ceil_div((long long)tiles_m * tiles_n, 8);
    const int lds_bytes = STAGES * (BigTile<TM, TN>::ROWS + BigTile<TM, TN>::WIDE) * BK * 2;
    static bool configured = false;     // per instantiation
    if (!configured) {
        hipError_t status = hipFuncSetAttribute((const void*)gemm_mfma_big_kernel<MODE, TO, TN, TM, STAGES, GROUPED>,
                                                hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
        if (status != hipSuccess) {
            fw_set_error("gemm_mfma_big: cannot reserve %d bytes of LDS: %s", lds_bytes, hipGetErrorString(status));
            return -1;
        }
        configured = true;
    }
    gemm_mfma_big_kernel<MODE, TO, TN, TM, STAGES, GROUPED><<<per_xcd * 8, 256, lds_bytes, stream>>>(
        (const uint16_t*)a, (const uint16_t*)w, bias, (TO*)out, M, N, K, tiles_m, tiles_n, per_xcd, N, groups);
    return 0;
}
template <int MODE, typename TO, int TN = 4, int TM = 4>
static int launch_big(const void* a, const void* w, const float* bias, void* out, int M, int N, int K, hipStream_t stream) {
    return launch_tiles<MODE, TO, TN, TM, BSTAGES, false>(a, w, bias, out, M, N, K, fw_ceil_div(M, BigTile<TM, TN>::ROWS), BigGroups(), stream);
}

// The grouped product of fw_grouped_gemm on tiles of 128 places by 256 rows of W, for K a multiple of 32 and a of less than 4 GB. Bound by
// the experts' weights from memory (600 MB for both products of 32 experts of 1,536 features: 127 us) and by tiles that an expert's last places fill partly.
// Two workgroups share a compute unit (three stages of 24 KB each), so that one multiplies while the other starts, ends or waits. 2,048 rows, 4 of 32
// experts, gated 1,536 over 2,048: 158 us; with four stages and one workgroup 175, on tiles of 256 places 186; through registers (moe.hip) 241.
bool fw_grouped_big_takes(int a_rows, int N, int K) { return K % BK == 0 && K <= BK_MOST && N <= BN_MOST && 2ll * a_rows * K <= 0xffff0000ll; }
int fw_launch_grouped_big(const void* a, const int32_t* place_row, const void* w, const int32_t* expert_begin, void* out, int gated, int places,
                          int experts, int N, int K, hipStream_t stream) {
    const BigGroups groups = {place_row, expert_begin, experts};
    const int tiles_m = places / 128 + (experts < places ? experts : places);       // at most: every expert's last tile may not be full
    // (what the product through registers, whose tiles have half the features, would refuse is refused here too)
    FW_REQUIRE((long long)tiles_m * fw_ceil_div(N, gated ? BT / 4 : BT / 2) < (1ll << 30), "grouped_gemm: too many tiles");
    if (gated) return launch_tiles<MB_SWIGLU, bf16_t, 4, 2, 3, true>(a, w, nullptr, out, places, N, K, tiles_m, groups, stream);
    return launch_tiles<MB_STORE, float, 4, 2, 3, true>(a, w, nullptr, out, places, N, K, tiles_m, groups, stream);
}

// The tile a storing or accumulating product is cut into: 256 or 128 rows by 256 or 192 columns,
// whichever takes the least time by this count: rounds of tiles over the chip's 256 compute units
// times the tile's area, a tile of 128 rows counting a quarter more than its area (it moves more
// bytes per flop). Gated products (SwiGLU) keep 256 x 256. (2,048 x 3,072 x 2,048: storing 50.9 -> 35.6 us with tiles of
// 128 x 192. Accumulating ones asked for each old value behind the store of the one before it and lost with twice the tiles; asked
// for a column of the tile at a time they gain as well.)
struct BigPlan {
    int rows, columns, tiles;
};
static BigPlan big_plan(int mode, int M, int N) {
    if (mode == MB_SWIGLU) return {BT, BT / 2, fw_ceil_div(M, BT) * fw_ceil_div(N, BT / 2)};
    BigPlan best = {0, 0, 0};
    long long best_cost = 0;
    for (int rows = BT; rows >= BT / 2; rows /= 2)
        for (int columns = BT; columns >= 192; columns -= 64) {
            const long long tiles = (long long)fw_ceil_div(M, rows) * fw_ceil_div(N, columns);
            const long long cost = fw_ceil_div(tiles, 256) * (rows / 32) * (columns / 32) * (rows == BT ? 4 : 5);
            if (best.tiles == 0 || cost < best_cost) {
                best = {rows, columns, (int)(tiles < (1ll << 30) ? tiles : (1ll << 30))};
                best_cost = cost;
            }
        }
    return best;
}

// How many tiles the kernel cuts a shape into, by the tile it will choose, and that tile's edges (the caller works out from them
// whether that fills the chip); 0 if the kernel does not take the shape (K must be a multiple of 32).
extern "C" int fw_gemm_mfma_big_plan(int mode, int M, int N, int K, int* rows, int* columns) {
    if (K <= 0 || K % BK || K > BK_MOST || M < 1 || N < 1 || N > BN_MOST) return 0;
    const BigPlan plan = big_plan(mode, M, N);
    if (rows) *rows = plan.rows;
    if (columns) *columns = plan.columns;
    return plan.tiles;
}

template <int MODE, typename TO>
static int launch_planned(const BigPlan& plan, const void* a, const void* w, const float* bias, void* out, int M, int N, int K,
                          hipStream_t stream) {
    if (plan.rows == BT)
        return plan.columns == BT ? launch_big<MODE, TO, 4, 4>(a, w, bias, out, M, N, K, stream)
                                  : launch_big<MODE, TO, 3, 4>(a, w, bias, out, M, N, K, stream);
    return plan.columns == BT ? launch_big<MODE, TO, 4, 2>(a, w, bias, out, M, N, K, stream)
                              : launch_big<MODE, TO, 3, 2>(a, w, bias, out, M, N, K, stream);
}

// Same contract as fw_gemm_mfma.
extern "C" int fw_gemm_mfma_big(const void* a, const void* w, const float* bias, void* out, int out_dtype, int mode,
                                int M, int N, int K, void* stream) {
    FW_REQUIRE(M >= 1 && N > 0 && K > 0 && K % BK == 0, "gemm_mfma_big: K (%d) must be a positive multiple of %d; M=%d N=%d", K, BK, M, N);
    FW_REQUIRE(mode >= 0 && mode <= 2, "gemm_mfma_big: unknown mode %d", mode);
    FW_REQUIRE(mode != MB_ACCUMULATE || out_dtype == FW_F32, "gemm_mfma_big: accumulation needs a float32 destination");
    FW_REQUIRE(mode != MB_SWIGLU || ((out_dtype == FW_BF16 || out_dtype == FW_BF16_GEGLU) && bias == nullptr), "gemm_mfma_big: SwiGLU stores bfloat16 and takes no bias");
    FW_REQUIRE(out_dtype == FW_F32 || out_dtype == FW_BF16 || (out_dtype == FW_BF16_GELU && mode == MB_STORE) || (out_dtype == FW_BF16_GEGLU && mode == MB_SWIGLU), "gemm_mfma_big: unknown out dtype %d", out_dtype);
    FW_REQUIRE(((uintptr_t)a % 16 == 0) && ((uintptr_t)w % 16 == 0), "gemm_mfma_big: operands must be 16-byte aligned");
    FW_REQUIRE((long long)fw_ceil_div(M, BT / 2) * fw_ceil_div(N, BT / 2) < (1ll << 30), "gemm_mfma_big: too many tiles");
    // rows too long for a lane's 32-bit places (8 MB of an operand, 4 MB of the output) go through registers, with 64-bit addresses
    if (K > BK_MOST || N > BN_MOST) return fw_gemm_mfma(a, w, bias, out, out_dtype, mode, M, N, K, stream);
    hipStream_t s = (hipStream_t)stream;
    const BigPlan plan = big_plan(mode, M, N);
    int status;
    if (mode == MB_SWIGLU && out_dtype == FW_BF16_GEGLU) status = launch_big<MB_SWIGLU, geglu_bf16_t>(a, w, nullptr, out, M, N, K, s);
    else if (mode == MB_SWIGLU) status = launch_big<MB_SWIGLU, bf16_t>(a, w, nullptr, out, M, N, K, s);
    else if (mode == MB_ACCUMULATE) status = launch_planned<MB_ACCUMULATE, float>(plan, a, w, bias, out, M, N, K, s);
    else if (out_dtype == FW_F32) status = launch_planned<MB_STORE, float>(plan, a, w, bias, out, M, N, K, s);
    else if (out_dtype == FW_BF16_GELU) status = launch_planned<MB_STORE, gelu_bf16_t>(plan, a, w, bias, out, M, N, K, s);
    else status = launch_planned<MB_STORE, bf16_t>(plan, a, w, bias, out, M, N, K, s);
    if (status != 0) return status;
    FW_LAUNCH_CHECK("gemm_mfma_big");
    return 0;
}
