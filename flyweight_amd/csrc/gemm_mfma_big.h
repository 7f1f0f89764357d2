// Tiled matrix product for long prompts and wide outputs: out[M][N] = a[M][K] . w[N][K]^T with
// 256 x 256 tiles. The 128 x 128 kernel beside this one moves 64 KB through a compute unit's
// vector memory path (64 bytes a clock) for every 1,024 clocks of MFMA work: at full MFMA rate
// the path would be busy all the time, and the kernel is bound by it at a third of the peak.
// Twice the tile edge halves the bytes per flop, in the memory path and in LDS alike:
//
//  * a workgroup of four waves computes 256 x 256; each wave a 128 x 128 quarter as 8 x 8 tiles of
//    v_mfma_f32_16x16x32_bf16, its 256 accumulators in the accumulation registers; one wave per
//    SIMD, so the overlap of loads, LDS reads and MFMAs is inside the wave. (The same products on
//    v_mfma_f32_32x32x16_bf16 move twice the accumulators per flop and draw more power: 8,192^3 at 1.45 GHz
//    against 1.6. Both give the same bits.);
//  * 256 x 64 slabs of both operands travel from global memory STRAIGHT into LDS
//    (buffer_load_dwordx4 .. lds: no staging registers, which the accumulators leave no room for),
//    two stages of a and three of w in all 160 KB, one barrier per slab; a row of a slab is a whole cache
//    line (slabs of 32 k ask L2 for every line in two halves: twice the requests, 11 of the 16 a clock that a
//    die's L2 takes); rows are not padded, their chunks are stored permuted against bank conflicts;
//  * workgroups are numbered so that each XCD works on a compact group of tiles.
//
// The same loop runs on smaller and on wider tiles, 64 to 256 rows by 128 to 320 columns: a round of tiles that the chip's 256 compute units
// are not full with is as long as a whole one, so the tile follows the shape. 2,048 rows by 3,072 features are 128 tiles of 256 x 192 but exactly 256 of
// 128 x 192; 2,048 x 4,608 gated over K 1,024 is 288 tiles of 256 x 256, two rounds and 55 us, but 232 of 256 x 320, one and 38; 1,111 x 2,048 over K 2,048 are
// 40 tiles of 256 x 256, 41 us with the launch, and 198 of 64 x 192, 21; 300 x 8,192 gated over K 2,048 42 us on 256 x 256 and 31 on 192 x 128. A smaller tile moves more bytes per flop
// through LDS and the memory path (which its six stages, or a second workgroup on the compute unit, keep busy), so it is used only where it fills the
// chip better: the caller compares the products' estimated times.
//
// Epilogues as the other products: store, add into the residual stream, SwiGLU
// (a tile holds as many gate as up features of the same columns; a lane holds both of an
// element). The experts' grouped product of a prompt runs in the same loop, its tiles numbered as grouped.h says. The reference's prompt GEMM is a 64x64 tile of plain FMAs without tensor cores
// (native/include/flyweight_v2_native_kernels.hpp:233-311).
#pragma once
#include "fw_common.h"
#include "fw_kernels.h"
#include "gemm_big.h"
#include "grouped.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

#define BT 256                  // tile edge (rows: of the tall tiles)
#define BK 32                   // k of one step of products: K is a multiple of it
#define BSLAB 64                // k of a slab, two steps
#define BLDS 163840             // bytes of LDS of a compute unit
#define BK_MOST (1 << 22)
#define BN_MOST (1 << 20)       // 256 rows of the output lie below BOUNDS
#define BOUNDS 0x80000000u
#define BGROUP_M 4
#define B_SLICES 8              // most slices of K

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
// The logistic function as exact as with expf and a division, without their cases (two prompts of four layers with 8,192 gated features over 2,048, 2,618 us: 10 us more
// than with the hardware's alone; with expf and a division 44): e^-|z| as 2^t (1 + rest) with the product's rounding in the rest, and one step of Newton's behind the reciprocal. Largest error, -8 to 8 / -20 to -8 / -86 to -20:
// 2^-22.6 / 2^-22.3 / 2^-22.6 of the value; expf and a division 2^-22.4 / 2^-22.4 / 2^-23.5; the hardware's exponential and reciprocal alone 2^-20.9 / 2^-19.9 / 2^-18.
__device__ __forceinline__ float sigmoid_big(float z) {
    const float x = fmaxf(-fabsf(z), -150.0f);                             // (2^t is zero from there on)
    const float t = x * 1.44269504f, rest = fmaf(x, 1.92596299e-8f, fmaf(x, 1.44269504f, -t));        // log2 e in two parts
    const float power = __builtin_amdgcn_exp2f(t), e = fmaf(power, rest * 0.693147181f, power);
    const float r = __builtin_amdgcn_rcpf(1.0f + e);
    return (z >= 0.0f ? 1.0f : e) * fmaf(fmaf(-(1.0f + e), r, 1.0f), r, r);
}
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
// behind the other, row by row or (tiled) all rows in operand tiles: a wave-wide load then takes a whole tile, lane for lane as an operand has it, and leaves it in LDS
// so. Both products of 32 experts of 1,536 features over 2,048, four a row, by rows / tiles: 600 rows 142 / 125 us, 2,048 rows 230 / 224. (Tiles asked for in the order of
// rows, 16 lanes of a load in 8 lines instead of 2: a prompt of 2,048 tokens with three such layers 2,120 -> 2,240 us.)
struct BigGroups {
    const int32_t *place_row, *begin;
    int experts;
    bool tiled;
};

// K cut over workgroups: `slices` of k_each, which meet in a workspace [slice][tile][product tile][thread][4] through a ticket a tile.
struct BigSlices {
    int slices, k_each;
    float* partials;
    int* counters;
};

// A gated product with this output type stores the unit with clamped halves (as fw_clamped_glu forms it) in bfloat16.
struct clamped_bf16_t {
    uint16_t bits;
};
struct BigUnit {
    float limit, alpha, shift;
};
template <typename TO> struct big_clamps { static constexpr bool value = false; };
template <> struct big_clamps<clamped_bf16_t> { static constexpr bool value = true; };

// A slab: 64 k of the tile's rows (an LDS row is 128 bytes, eight 16-byte chunks). Chunk
// c of a row lies in slot c ^ swap(row): a read of 16 rows by four chunks goes in groups of 16 lanes, 0-3, 12-15 and 20-27, then the 16
// others of the first 32, and every group covers all 64 banks once.
__device__ __forceinline__ int chunk_swap(int row) { return (row >> 1) & 7; }

template <int TM, int TN, int EACH_CU>
struct BigTile {
    static constexpr int ROWS = 2 * TM * 32;               // rows of a tile
    static constexpr int WIDE = 2 * TN * 32;               // columns of a tile
    static constexpr int A_SLAB = ROWS * BSLAB * 2, W_SLAB = WIDE * BSLAB * 2;     // bytes
    static constexpr int A_LOADS = A_SLAB / 4096;          // wave-wide loads per wave for a slab of a (1,024 bytes each)
    static constexpr int W_LOADS = W_SLAB / 4096;          // and for a slab of w
    static constexpr int SLAB_LOADS = A_LOADS + W_LOADS;   // and for a slab of both operands
    // slabs in LDS, the one that is multiplied among them: as many of both as fit, and one more of w if it fits beside them
    static constexpr int LDS_MOST = BLDS / EACH_CU, MOST_STAGES = TM * TN <= 4 ? 6 : 4;
    static constexpr int A_STAGES = LDS_MOST / (A_SLAB + W_SLAB) < MOST_STAGES ? LDS_MOST / (A_SLAB + W_SLAB) : MOST_STAGES;
    static constexpr int W_STAGES = A_STAGES < 3 && A_STAGES * A_SLAB + (A_STAGES + 1) * W_SLAB <= LDS_MOST ? A_STAGES + 1 : A_STAGES;
    static constexpr int LDS = A_STAGES * A_SLAB + W_STAGES * W_SLAB;
    // whether w is asked for together with a, behind the products that follow a slab's last read: where w has two stages (asked for a step later its
    // slab would have one step to arrive)
    static constexpr bool TOGETHER = W_STAGES == 2;
};

// K must be a multiple of BK (the loads go straight to LDS: nothing can be zeroed on the way), and at most BK_MOST (a
// lane's place in a tile's 256 rows is 32 bits, as it is in the output: N at most BN_MOST).
//
// Bound by the matrix cores at the clock that their power leaves (1.5 to 1.9 GHz): 77 % of a wave's cycles in MFMAs at 8,192^3, the rest at a tile's
// start and end and where a slab's loads are waited for. Against slabs of 32 k on v_mfma_f32_32x32x16_bf16: 2,048 x 8,192 gated x 2,048 120.8 -> 104.7 us
// (1,310 TFLOP/s), storing 2,048 x 6,144 x 2,048 52.8 -> 44.0, 2,048 x 3,072 x 2,048 30.7 -> 25.4, 1,111 x 16,384 x 2,048 90.4 -> 79.0, 8,192^3 1,254 -> 1,470
// TFLOP/s. Where the loads stand among the MFMAs (behind every second to every eighth) changed nothing; two stages of w instead of three cost 1 to 8 %.
// TN: 32-column pairs of product tiles per wave, 2 (128 columns a tile) to 5 (320). TM: 32-row pairs of product tiles per wave, 1 (64 rows a tile) to
// 4. EACH_CU: workgroups on a compute unit.
template <int MODE, typename TO, int TN, int TM, bool GROUPED, bool SPLIT, int EACH_CU>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(EACH_CU, EACH_CU))) void gemm_mfma_big_kernel(
    const uint16_t* __restrict__ a, const uint16_t* __restrict__ w, const float* __restrict__ bias,
    TO* __restrict__ out, int M, int N, int K, int tiles_m, int tiles_n, int per_xcd, int up_offset, const BigGroups groups, const BigSlices cut, const BigUnit halves) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];      // [A_STAGES slabs of a][W_STAGES slabs of w]
    typedef BigTile<TM, TN, EACH_CU> Tile;
    constexpr int ROWS = Tile::ROWS, WIDE = Tile::WIDE, A_SLAB = Tile::A_SLAB, W_SLAB = Tile::W_SLAB, A_STAGES = Tile::A_STAGES, W_STAGES = Tile::W_STAGES;
    constexpr int A_LOADS = Tile::A_LOADS, W_LOADS = Tile::W_LOADS, SLAB_LOADS = Tile::SLAB_LOADS;
    constexpr bool TOGETHER = Tile::TOGETHER;
    constexpr int PARTS = BSLAB / BK, CHUNKS = BSLAB / 8, LOAD_ROWS = 64 / CHUNKS;      // steps of a slab, chunks of a row, rows of a wave-wide load
    static_assert(PARTS == 2, "the loop has two steps a slab");
    constexpr int features = MODE == MB_SWIGLU ? WIDE / 2 : WIDE;       // a gated tile holds as many gate as up rows
    int m0, n0, k_first = 0, k_length = K;
    const int32_t* groups_rows = nullptr;
    const bool tiled = GROUPED && groups.tiled;
    size_t w_row = 0;                                       // of w: this expert's first
    int slice = 0, tile_number = 0;
    if constexpr (GROUPED) {
        const GroupedTile tile = grouped_tile(groups.begin, groups.experts, ROWS, tiles_n);
        const int expert = tile.expert;
        if (expert < 0) return;
        m0 = tile.row_tile * ROWS;
        n0 = tile.column_tile * features;
        const int first = groups.begin[expert];
        M = groups.begin[expert + 1] - first;           // rows of this expert: places first .. first + M - 1
        w_row = (size_t)expert * (MODE == MB_SWIGLU ? 2 : 1) * N;
        out += (size_t)first * N;
        if (groups.place_row) groups_rows = groups.place_row + first;
        else a += (size_t)first * K;
    } else {
        const int total = tiles_m * tiles_n;
        int logical = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
        if (logical >= total * (SPLIT ? cut.slices : 1)) return;
        if constexpr (SPLIT) {              // slice by slice: a die's workgroups share what they read of a and w
            slice = logical / total;
            logical -= slice * total;
            tile_number = logical;
            k_first = slice * cut.k_each;
            k_length = K - k_first < cut.k_each ? K - k_first : cut.k_each;
        }
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
    // l * 16: 8 rows of 128 bytes (16 of 64). Rows are not padded; instead the chunks of a row are
    // stored permuted (chunk_swap): lane l therefore ASKS for the chunk whose slot it fills. Addresses are a base that the wave shares (the tile's first row; of a gated
    // product's w the first gate or up row: a wave's loads of w are all of one kind), a 32-bit
    // offset of the lane, and the slab's offset in a scalar register: a slab costs no vector arithmetic.
    const int w_part = MODE == MB_SWIGLU && wave >= 2 ? 1 : 0;
    const int w_first = MODE == MB_SWIGLU ? w_part * up_offset + n0 : n0;
    const uint16_t* a_base = GROUPED && groups_rows ? a : a + (size_t)m0 * K;
    w_row += w_first;
    const uint16_t* w_base = w + (tiled ? w_row & ~(size_t)15 : w_row) * K;
    const int w_step = tiled ? 2048 : BSLAB * 2;            // bytes of w from a slab to the next
    uint32_t a_at[A_LOADS], w_at[W_LOADS];
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) {
        const int row = (wave * A_LOADS + i) * LOAD_ROWS + lane / CHUNKS;
        const int chunk = (lane % CHUNKS) ^ chunk_swap(row);
        uint32_t from = row < M - m0 ? row : M - m0 - 1;        // rows past the end are computed and dropped
        if (GROUPED && groups_rows) from = groups_rows[m0 + (int)from];
        a_at[i] = from * (uint32_t)(2 * K) + chunk * 16;
    }
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i) {
        const int load = wave * W_LOADS + i, row = tiled ? (load >> 1) * 16 + (lane & 15) : load * LOAD_ROWS + lane / CHUNKS;
        const int of_part = MODE == MB_SWIGLU ? row - w_part * features : row;
        const uint32_t from = of_part < N - n0 ? of_part : N - n0 - 1;
        if (tiled) {
            const uint32_t of_tiles = (uint32_t)(w_row & 15) + from;
            w_at[i] = (of_tiles >> 4) * (uint32_t)(32 * K) + (load & 1) * 1024 + (lane >> 4) * 256 + (of_tiles & 15) * 16;
        } else {
            w_at[i] = from * (uint32_t)(2 * K) + ((lane % CHUNKS) ^ chunk_swap(row)) * 16;
        }
    }
    const fw_buffer a_rows = fw_make_buffer(a_base + k_first), w_rows = fw_make_buffer(w_base + k_first);
    // This wave's loads for a slab of either operand, into the stage at `stage`. A last slab of half the length has no upper
    // chunks: the lower ones are read again in their place and never used.
    const int whole = k_length / BSLAB, slabs = (k_length + BSLAB - 1) / BSLAB;
    auto request_a = [&](int stage, int slab, int i) { fw_buffer_to_lds(a_rows, lds + stage + (wave * A_LOADS + i) * 1024, a_at[i], slab * (BSLAB * 2)); };
    auto request_w = [&](int stage, int slab, int i) { fw_buffer_to_lds(w_rows, lds + stage + (wave * W_LOADS + i) * 1024, w_at[i], slab * w_step); };
    auto upper = [&](int first_row) { return ((lane % CHUNKS) ^ chunk_swap(first_row + lane / CHUNKS)) >= CHUNKS / 2; };
    auto request_slab_a = [&](int stage, int slab) {
#pragma unroll
        for (int i = 0; i < A_LOADS; ++i) {
            if (slab >= whole && upper((wave * A_LOADS + i) * LOAD_ROWS)) a_at[i] -= BK * 2;
            request_a(stage, slab, i);
        }
    };
    auto request_slab_w = [&](int stage, int slab) {
#pragma unroll
        for (int i = 0; i < W_LOADS; ++i) {
            if (slab >= whole && (tiled ? (wave * W_LOADS + i) & 1 : upper((wave * W_LOADS + i) * LOAD_ROWS))) w_at[i] -= tiled ? 1024 : BK * 2;
            request_w(stage, slab, i);
        }
    };

    constexpr int TA = 2 * TM, TB = 2 * TN;     // 16-row and 16-column product tiles of the wave
    f32x4 acc[TA][TB];
#pragma unroll
    for (int i = 0; i < TA; ++i)
#pragma unroll
        for (int j = 0; j < TB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // this wave's rows of the a slab, and its rows of the w slab: for SwiGLU the columns of a wave
    // are 16 TN gate features (tiles 0 to TN - 1) and the up features of the same columns (the tiles behind).
    // Every row this lane reads is (lane % 16) plus a multiple of 16: one permutation for all
    int slot[PARTS];
#pragma unroll
    for (int t = 0; t < PARTS; ++t) slot[t] = ((4 * t + (lane >> 4)) ^ chunk_swap(lane & 15)) * 16;
    const int a_row0 = wm * (TM * 32) + (lane & 15), b_tile0 = wn * (MODE == MB_SWIGLU ? TN : TN * 2);
    int b_at[PARTS];                                        // of this lane's operand of the wave's first column tile; the others lie 2,048 bytes on each
#pragma unroll
    for (int t = 0; t < PARTS; ++t) b_at[t] = b_tile0 * (16 * BSLAB * 2) + (tiled ? t * 1024 + lane * 16 : slot[t] + (lane & 15) * (BSLAB * 2));

    // operand registers of one step: the wave's row tiles of a and column tiles of w
    struct Operands {
        bf16x8 fa[TA], fb[TB];
    };
    constexpr int MFMAS = TA * TB, READS = TA + TB;
    constexpr int W_FIRST = A_STAGES * A_SLAB, W_END = W_FIRST + W_STAGES * W_SLAB;
    // the stages of slab s and the one behind it, and of w the one ahead of it
    int a_now = 0, a_then = A_SLAB, w_now = W_FIRST, w_then = W_FIRST + W_SLAB, w_before = W_END - W_SLAB;
    auto advance = [&]() {
        a_now = a_then;
        a_then = a_then + A_SLAB < W_FIRST ? a_then + A_SLAB : 0;
        w_before = w_now;
        w_now = w_then;
        w_then = w_then + W_SLAB < W_END ? w_then + W_SLAB : W_FIRST;
    };
    auto read_one = [&](Operands& f, int a_stage, int w_stage, int part, int which) {
        if (which < TA) {
            f.fa[which] = *reinterpret_cast<const bf16x8*>(lds + a_stage + slot[part] + (a_row0 + 16 * which) * (BSLAB * 2));
        } else {
            const int j = which - TA, row = MODE == MB_SWIGLU ? (j / TN) * features + (j % TN) * 16 : j * 16;
            f.fb[j] = *reinterpret_cast<const bf16x8*>(lds + w_stage + b_at[part] + row * (BSLAB * 2));
        }
    };
    auto read = [&](Operands& f, int a_stage, int w_stage, int part) {
#pragma unroll
        for (int u = 0; u < READS; ++u) read_one(f, a_stage, w_stage, part, u);
    };
    // product tile number `which`, row by row, every second row backwards
    auto multiply_one = [&](const Operands& f, int which) {
        const int i = which / TB, j = i & 1 ? TB - 1 - which % TB : which % TB;
        if (i * TB + j < 64) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(f.fa[i]), "v"(f.fb[j]));
        else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc[i][j]) : "v"(f.fa[i]), "v"(f.fb[j]));      // (256 accumulation registers)
    };
    auto multiply = [&](const Operands& f) {
#pragma unroll
        for (int u = 0; u < MFMAS; ++u) multiply_one(f, u);
    };
    // Tells the compiler that these operands are needed HERE, so that it waits for their LDS reads
    // before the next reads are issued and not, for all reads together, in front of the MFMAs.
    auto arrived = [&](const Operands& f) {
#pragma unroll
        for (int i = 0; i < TA; i += 2) asm volatile("" ::"v"(f.fa[i]), "v"(f.fa[i + 1]));
#pragma unroll
        for (int j = 0; j < TB; j += 2) asm volatile("" ::"v"(f.fb[j]), "v"(f.fb[j + 1]));
        // two wait states between moves that have written an operand or an accumulator and the product that reads it: the compiler
        // does not see a product in the assembly
        asm volatile("s_nop 1");
    };
    // waits until at most `slabs` of this wave's requested slabs (of both operands, or of w alone where w has a stage more) are still on their way
    constexpr int EACH = W_STAGES > A_STAGES ? W_LOADS : SLAB_LOADS;
    auto wait_for_all_but = [&](int slabs) {
        if (slabs >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * EACH) : "memory");
        else if (slabs == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(1 * EACH) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };

    // With one wave per SIMD nothing else hides the latency of LDS: the operands of a step are read behind the MFMAs of the step
    // before it. Ahead of a slab's last step the wave makes sure that the next slab has landed (its own loads: vmcnt; everybody's: the
    // barrier), which also tells that every wave has read slab s. Its stages then take the slabs that come A_STAGES and W_STAGES later:
    // that of a behind the MFMAs of the slab's last step, that of w behind those of the next slab's first.
    for (int u = 0; u < W_STAGES - 1; ++u) {
        if (u < slabs) request_slab_a(u * A_SLAB, u);
        if (u < slabs) request_slab_w(W_FIRST + u * W_SLAB, u);
    }
    if (A_STAGES == W_STAGES && A_STAGES <= slabs) request_slab_a((A_STAGES - 1) * A_SLAB, A_STAGES - 1);
    if (TOGETHER && W_STAGES <= slabs) request_slab_w(W_END - W_SLAB, W_STAGES - 1);
    if (slabs >= W_STAGES) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((A_STAGES - 1) * A_LOADS + (W_STAGES - (TOGETHER ? 1 : 2)) * W_LOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    Operands f0, f1;
    read(f0, a_now, w_now, 0);
    int s = 0;
    // two MFMAs (32 clocks) to a read: four waves that read at once keep LDS busy for as long
    constexpr int READ_GAP = 2 * READS <= MFMAS ? 2 : 1, A_GAP = MFMAS / A_LOADS, W_GAP = MFMAS / W_LOADS;
    auto landed = [&](const Operands& f) {
        arrived(f);                                         // slab s has been read
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((W_STAGES - 2) * EACH) : "memory");   // slab s + 1 has landed; those behind it may still fly
        __builtin_amdgcn_s_barrier();
    };
    while (s + A_STAGES < whole) {
        arrived(f0);
#pragma unroll
        for (int u = 0; u < MFMAS; ++u) {
            if (u % READ_GAP == 0 && u / READ_GAP < READS) read_one(f1, a_now, w_now, 1, u / READ_GAP);
            if (!TOGETHER && u % W_GAP == 0 && u / W_GAP < W_LOADS) request_w(w_before, s + W_STAGES - 1, u / W_GAP);
            multiply_one(f0, u);
            __builtin_amdgcn_sched_barrier(0);
        }
        landed(f1);
#pragma unroll
        for (int u = 0; u < MFMAS; ++u) {
            if (u % READ_GAP == 0 && u / READ_GAP < READS) read_one(f0, a_then, w_then, 0, u / READ_GAP);
            if (u % A_GAP == 0 && u / A_GAP < A_LOADS) request_a(a_now, s + A_STAGES, u / A_GAP);
            if (TOGETHER && u % W_GAP == W_GAP / 2 && u / W_GAP < W_LOADS) request_w(w_now, s + W_STAGES, u / W_GAP);
            multiply_one(f1, u);
            __builtin_amdgcn_sched_barrier(0);
        }
        advance();
        ++s;
    }
    // the last slabs: asking for what is left to ask for; one of two steps may have half the length
    for (; s < slabs; ++s) {
        const int ahead = (slabs < s + W_STAGES ? slabs : s + W_STAGES) - (s + 2);      // slabs behind s + 1 that have been asked for
        arrived(f0);
        if (s < whole) read(f1, a_now, w_now, 1);
        if (!TOGETHER && s + W_STAGES - 1 < slabs) request_slab_w(w_before, s + W_STAGES - 1);
        multiply(f0);
        __builtin_amdgcn_sched_barrier(0);
        arrived(f1);
        if (s + 1 < slabs) {
            wait_for_all_but(ahead);
            __builtin_amdgcn_s_barrier();
            read(f0, a_then, w_then, 0);
            if (s + A_STAGES < slabs) request_slab_a(a_now, s + A_STAGES);
            if (TOGETHER && s + W_STAGES < slabs) request_slab_w(w_now, s + W_STAGES);
        }
        if (s < whole) multiply(f1);
        __builtin_amdgcn_sched_barrier(0);
        advance();
    }
    fw_mfma_drain();     // branches follow that lead to code reading the accumulators

    // A slice's sums leave past the die's cache (device scope). Every wave waits until its own are acknowledged, then one thread takes the
    // ticket, and the last workgroup of the tile adds the slices in their order.
    if constexpr (SPLIT) {
        const int total = tiles_m * tiles_n;
        constexpr int TILE_BYTES = ROWS * WIDE * 4;
        auto left_by = [&](int of) { return fw_make_buffer(cut.partials + ((size_t)of * total + tile_number) * (TILE_BYTES / 4), TILE_BYTES); };
        const fw_buffer mine = left_by(slice);
#pragma unroll
        for (int u = 0; u < MFMAS; ++u) fw_buffer_store_device(mine, tid * 16, u * 4096, acc[u / TB][u % TB]);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        int* ticket = reinterpret_cast<int*>(lds);
        if (tid == 0) *ticket = __hip_atomic_fetch_add(&cut.counters[tile_number], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*ticket != cut.slices - 1) return;
        if (tid == 0) __hip_atomic_store(&cut.counters[tile_number], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // Its own sums it still holds; those of the others are asked for as many together as there are registers for.
        constexpr int HELD = MFMAS <= 12 ? 3 : MFMAS <= 16 ? 2 : 1;
        f32x4 sum[TA][TB];
        bool started = false;
        auto add = [&](const f32x4 (&part)[TA][TB]) {
#pragma unroll
            for (int u = 0; u < MFMAS; ++u) sum[u / TB][u % TB] = started ? sum[u / TB][u % TB] + part[u / TB][u % TB] : part[u / TB][u % TB];
            started = true;
        };
        for (int first = 0; first < cut.slices - 1; first += HELD) {
            f32x4 part[HELD][TA][TB];
#pragma unroll
            for (int h = 0; h < HELD; ++h) {
                const int other = first + h;
                if (other < cut.slices - 1) {
                    const fw_buffer theirs = left_by(other < slice ? other : other + 1);
#pragma unroll
                    for (int u = 0; u < MFMAS; ++u) part[h][u / TB][u % TB] = fw_buffer_load_device(theirs, tid * 16, u * 4096);
                }
            }
#pragma unroll
            for (int h = 0; h < HELD; ++h) {
                if (first + h < cut.slices - 1) {
                    if (first + h == slice) add(acc);
                    add(part[h]);
                }
            }
        }
        if (slice == cut.slices - 1) add(acc);
#pragma unroll
        for (int u = 0; u < MFMAS; ++u) acc[u / TB][u % TB] = sum[u / TB][u % TB];
    }

    // D layout of the 16x16 product: lane holds column lane % 16, register r is row 4 * (lane / 16) + r. Two neighbouring
    // column tiles swap every second 16 lanes, so that a lane holds column lane % 32 of the pair and eight rows
    // 8 * (lane / 32) + u of the row tile: a store then covers whole runs of 32 columns.
    const int col = lane & 31, row_base = (lane >> 5) * 8;
    auto paired = [](const float (&left)[4], const float (&right)[4], float (&rows)[8]) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const auto swapped = __builtin_amdgcn_permlane16_swap(__float_as_uint(left[r]), __float_as_uint(right[r]), false, false);
            const uint32_t upper = swapped[0], lower = swapped[1];
            rows[r] = __uint_as_float(upper);
            rows[4 + r] = __uint_as_float(lower);
        }
    };
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
    auto gated = [&](float g, float u) {
        if constexpr (big_clamps<TO>::value) {
            g = fminf(g, halves.limit);
            u = fminf(fmaxf(u, -halves.limit), halves.limit);
            return g * sigmoid_big(halves.alpha * g) * (u + halves.shift);
        } else {
            return fw_gate_of<TO>(g, unit) * u;
        }
    };
    const uint32_t first_row = (uint32_t)(wm * (TM * 32) + row_base);      // of this lane, of the tile
    // the eight rows of row tile i and pair j of column tiles that this lane holds: gated, or with the bias
    constexpr int SHARE = MODE == MB_SWIGLU ? TN * 16 : TN * 32, PAIRS = SHARE / 32;       // columns of the output that a wave holds
    auto values = [&](int i, int j, float b, float (&rows)[8]) {
        float left[4], right[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if constexpr (MODE == MB_SWIGLU) {
                left[r] = gated(acc[i][2 * j][r], acc[i][2 * j + TN][r]);
                right[r] = gated(acc[i][2 * j + 1][r], acc[i][2 * j + 1 + TN][r]);
            } else {
                left[r] = acc[i][2 * j][r];
                right[r] = acc[i][2 * j + 1][r];
            }
        }
        paired(left, right, rows);
        if constexpr (MODE != MB_SWIGLU)
#pragma unroll
            for (int u = 0; u < 8; ++u) rows[u] = fw_before_store<TO>(rows[u] + b);
    };
    // A gated tile of an odd number of column tiles a wave: its last one has no neighbour, and lanes hold column lane % 16 and rows 4 * (lane / 16) + r of it.
    constexpr bool LONE = SHARE % 32 != 0;
    const int lone_column = wn * SHARE + PAIRS * 32 + (lane & 15);
    const uint32_t lone_row = (uint32_t)(wm * (TM * 32) + (lane >> 4) * 4);
    auto lone_values = [&](int i, float (&rows)[4]) {
#pragma unroll
        for (int r = 0; r < 4; ++r) rows[r] = gated(acc[i][TN - 1][r], acc[i][2 * TN - 1][r]);
    };
    if (SIZE == 4 || ((N & 1) == 0 && (uintptr_t)out % 4 == 0)) {
#pragma unroll
        for (int j = 0; j < PAIRS; ++j) {
            const int c = wn * SHARE + j * 32 + col;        // column of the tile
            const bool there = n0 + c < N;
            const float b = MODE != MB_SWIGLU && bias && there ? bias[n0 + c] : 0.0f;
            if constexpr (SIZE == 4) {
                const uint32_t at = there ? first_row * row_step + c * 4 : BOUNDS;
                float old[MODE == MB_ACCUMULATE ? TA * 8 : 1];
                if constexpr (MODE == MB_ACCUMULATE) {
#pragma unroll
                    for (int u = 0; u < TA * 8; ++u) old[u] = fw_buffer_load_float(to, at + (uint32_t)((u >> 3) * 16 + (u & 7)) * row_step);
                }
#pragma unroll
                for (int i = 0; i < TA; ++i) {
                    float rows[8];
                    values(i, j, b, rows);
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        if (MODE == MB_ACCUMULATE) rows[u] += old[i * 8 + u];
                        fw_buffer_store(to, at + (uint32_t)(i * 16 + u) * row_step, __builtin_bit_cast(uint32_t, rows[u]));
                    }
                }
            } else {
                const uint32_t at = there ? (first_row + (odd ? 1 : 0)) * row_step + (c & ~1) * 2 : BOUNDS;
#pragma unroll
                for (int i = 0; i < TA; ++i) {
                    float rows[8];
                    values(i, j, b, rows);
#pragma unroll
                    for (int u = 0; u < 8; u += 2) {
                        const float got = from_neighbour(odd ? rows[u] : rows[u + 1]);
                        const uint32_t word = odd ? pack_bf16x2(got, rows[u + 1]) : pack_bf16x2(rows[u], got);
                        fw_buffer_store(to, at + (uint32_t)(i * 16 + u) * row_step, word);
                    }
                }
            }
        }
        if constexpr (LONE) {
            const uint32_t at = n0 + lone_column < N ? (lone_row + (odd ? 1 : 0)) * row_step + (lone_column & ~1) * 2 : BOUNDS;
#pragma unroll
            for (int i = 0; i < TA; ++i) {
                float rows[4];
                lone_values(i, rows);
#pragma unroll
                for (int u = 0; u < 4; u += 2) {
                    const float got = from_neighbour(odd ? rows[u] : rows[u + 1]);
                    const uint32_t word = odd ? pack_bf16x2(got, rows[u + 1]) : pack_bf16x2(rows[u], got);
                    fw_buffer_store(to, at + (uint32_t)(i * 16 + u) * row_step, word);
                }
            }
        }
        return;
    }
    // Two bytes an element, and rows of an odd length or an output at an odd place: every element leaves by itself, just as free of branches
    // (with two an element 5,532 x 83 x 608 took 19.0 us against 11.5, 1,300 x 3,071 x 1,024 25.7 against 18.3).
    if constexpr (SIZE == 2) {
#pragma unroll
        for (int j = 0; j < PAIRS; ++j) {
            const int c = wn * SHARE + j * 32 + col;
            const bool there = n0 + c < N;
            const float b = MODE != MB_SWIGLU && bias && there ? bias[n0 + c] : 0.0f;
            const uint32_t at = there ? first_row * row_step + c * 2 : BOUNDS;
#pragma unroll
            for (int i = 0; i < TA; ++i) {
                float rows[8];
                values(i, j, b, rows);
#pragma unroll
                for (int u = 0; u < 8; ++u) fw_buffer_store(to, at + (uint32_t)(i * 16 + u) * row_step, float_to_bf16_bits(rows[u]));
            }
        }
        if constexpr (LONE) {
            const uint32_t at = n0 + lone_column < N ? lone_row * row_step + lone_column * 2 : BOUNDS;
#pragma unroll
            for (int i = 0; i < TA; ++i) {
                float rows[4];
                lone_values(i, rows);
#pragma unroll
                for (int u = 0; u < 4; ++u) fw_buffer_store(to, at + (uint32_t)(i * 16 + u) * row_step, float_to_bf16_bits(rows[u]));
            }
        }
    }
}

template <int MODE, typename TO, int TN, int TM, bool GROUPED, bool SPLIT, int EACH_CU>
static int launch_tiles(const void* a, const void* w, const float* bias, void* out, int M, int N, int K, int tiles_m, const BigGroups& groups,
                        hipStream_t stream, const BigSlices& cut = BigSlices(), const BigUnit& halves = BigUnit()) {
    const int tiles_n = fw_ceil_div(N, BigTile<TM, TN, EACH_CU>::WIDE / (MODE == MB_SWIGLU ? 2 : 1));
    const int per_xcd = fw_ceil_div((long long)tiles_m * tiles_n * (SPLIT ? cut.slices : 1), 8);
    const int lds_bytes = BigTile<TM, TN, EACH_CU>::LDS;
    static bool configured = false;     // per instantiation
    if (!configured) {
        hipError_t status = hipFuncSetAttribute((const void*)gemm_mfma_big_kernel<MODE, TO, TN, TM, GROUPED, SPLIT, EACH_CU>,
                                                hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
        if (status != hipSuccess) {
            fw_set_error("gemm_mfma_big: cannot reserve %d bytes of LDS: %s", lds_bytes, hipGetErrorString(status));
            return -1;
        }
        configured = true;
    }
    gemm_mfma_big_kernel<MODE, TO, TN, TM, GROUPED, SPLIT, EACH_CU><<<per_xcd * 8, 256, lds_bytes, stream>>>(
        (const uint16_t*)a, (const uint16_t*)w, bias, (TO*)out, M, N, K, tiles_m, tiles_n, per_xcd, N, groups, cut, halves);
    return 0;
}

// A product on the tile that the call names.
template <int MODE, typename TO, int TN, int TM, int EACH_CU, bool SPLIT>
static int launch_big(const BigCall& c) {
    const BigSlices cut = {c.slices, c.k_each, c.partials, c.counters};
    return launch_tiles<MODE, TO, TN, TM, false, SPLIT, EACH_CU>(c.a, c.w, c.bias, c.out, c.M, c.N, c.K, fw_ceil_div(c.M, TM * 64), BigGroups(), c.stream, cut, {c.limit, c.alpha, c.shift});
}
