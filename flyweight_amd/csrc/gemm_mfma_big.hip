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
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

#define BT 256                  // tile edge (rows: of the tall tiles)
#define BK 32                   // k of one step of products: K is a multiple of it
#define BLDS 163840             // bytes of LDS of a compute unit
#define BK_MOST (1 << 22)
#define BN_MOST (1 << 20)       // 256 rows of the output lie below BOUNDS
#define BOUNDS 0x80000000u
#define BGROUP_M 4
#define B_LOADS 8               // most wave-wide loads (1,024 bytes) per wave per operand per slab

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

// K cut over workgroups: `slices` of k_each, which meet in a workspace [slice][tile][product tile][thread][4] through a ticket a tile.
struct BigSlices {
    int slices, k_each;
    float* partials;
    int* counters;
};

// A slab: 64 k of the tile's rows (an LDS row is 128 bytes, eight 16-byte chunks), or 32 where two workgroups share a compute unit. Chunk
// c of a row lies in slot c ^ swap(row): a read of 16 rows by four chunks goes in groups of 16 lanes, 0-3, 12-15 and 20-27, then the 16
// others of the first 32, and every group covers all 64 banks once.
template <int DEPTH>
__device__ __forceinline__ int chunk_swap(int row) {
    if (DEPTH == 64) return (row >> 1) & 7;
    const int low = (row >> 2) & 1, high = (row >> 3) & 1;      // 0, 2, 3, 1 for four rows each
    return (low ^ high) * 2 + high;
}

template <int TM, int TN, int DEPTH>
struct BigTile {
    static constexpr int ROWS = 2 * TM * 32;               // rows of a tile
    static constexpr int WIDE = 2 * TN * 32;               // columns of a tile
    static constexpr int A_SLAB = ROWS * DEPTH * 2, W_SLAB = WIDE * DEPTH * 2;     // bytes
    static constexpr int A_LOADS = A_SLAB / 4096;          // wave-wide loads per wave for a slab of a (1,024 bytes each)
    static constexpr int W_LOADS = W_SLAB / 4096;          // and for a slab of w
    static constexpr int SLAB_LOADS = A_LOADS + W_LOADS;   // and for a slab of both operands
    // slabs in LDS, the one that is multiplied among them: as many of both as fit, and one more of w if it fits beside them
    static constexpr int LDS_MOST = DEPTH == 64 ? BLDS : BLDS / 2;
    static constexpr int A_STAGES = LDS_MOST / (A_SLAB + W_SLAB) < 4 ? LDS_MOST / (A_SLAB + W_SLAB) : 4;
    static constexpr int W_STAGES = A_STAGES < 3 && A_STAGES * A_SLAB + (A_STAGES + 1) * W_SLAB <= LDS_MOST ? A_STAGES + 1 : A_STAGES;
    static constexpr int LDS = A_STAGES * A_SLAB + W_STAGES * W_SLAB;
};

// K must be a multiple of BK (the loads go straight to LDS: nothing can be zeroed on the way), and at most BK_MOST (a
// lane's place in a tile's 256 rows is 32 bits, as it is in the output: N at most BN_MOST).
//
// Bound by the matrix cores at the clock that their power leaves (1.5 to 1.9 GHz): 77 % of a wave's cycles in MFMAs at 8,192^3, the rest at a tile's
// start and end and where a slab's loads are waited for. Against slabs of 32 k on v_mfma_f32_32x32x16_bf16: 2,048 x 8,192 gated x 2,048 120.8 -> 104.7 us
// (1,310 TFLOP/s), storing 2,048 x 6,144 x 2,048 52.8 -> 44.0, 2,048 x 3,072 x 2,048 30.7 -> 25.4, 1,111 x 16,384 x 2,048 90.4 -> 79.0, 8,192^3 1,254 -> 1,470
// TFLOP/s. Where the loads stand among the MFMAs (behind every second to every eighth) changed nothing; two stages of w instead of three cost 1 to 8 %.
// TN: 32-column pairs of product tiles per wave, 4 (a 256 x 256 tile) or 3 (256 x 192: a width of 6,144
// features gives 192 tiles of 256 columns for 256 compute units, but exactly 256 tiles of 192).
// TM: 32-row pairs of product tiles per wave, 4 (256 rows a tile) or 2 (128 rows). DEPTH: k of a slab, see BigTile.
template <int MODE, typename TO, int TN, int TM, int DEPTH, bool GROUPED, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DEPTH == 32 ? 2 : 1, DEPTH == 32 ? 2 : 1))) void gemm_mfma_big_kernel(
    const uint16_t* __restrict__ a, const uint16_t* __restrict__ w, const float* __restrict__ bias,
    TO* __restrict__ out, int M, int N, int K, int tiles_m, int tiles_n, int per_xcd, int up_offset, const BigGroups groups, const BigSlices cut) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];      // [A_STAGES slabs of a][W_STAGES slabs of w]
    typedef BigTile<TM, TN, DEPTH> Tile;
    constexpr int ROWS = Tile::ROWS, WIDE = Tile::WIDE, A_SLAB = Tile::A_SLAB, W_SLAB = Tile::W_SLAB, A_STAGES = Tile::A_STAGES, W_STAGES = Tile::W_STAGES;
    constexpr int A_LOADS = Tile::A_LOADS, W_LOADS = Tile::W_LOADS, SLAB_LOADS = Tile::SLAB_LOADS;
    constexpr int PARTS = DEPTH / BK, CHUNKS = DEPTH / 8, LOAD_ROWS = 64 / CHUNKS;      // steps of a slab, chunks of a row, rows of a wave-wide load
    const int features = MODE == MB_SWIGLU ? BT / 2 : WIDE;
    static_assert(MODE != MB_SWIGLU || TN == 4, "the gated tile holds 128 gate and 128 up rows");
    int m0, n0, k_first = 0, k_length = K;
    const int32_t* groups_rows = nullptr;
    int slice = 0, tile_number = 0;
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
    const uint16_t* w_base = w + (size_t)w_first * K;
    uint32_t a_at[A_LOADS], w_at[B_LOADS];
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) {
        const int row = (wave * A_LOADS + i) * LOAD_ROWS + lane / CHUNKS;
        const int chunk = (lane % CHUNKS) ^ chunk_swap<DEPTH>(row);
        uint32_t from = row < M - m0 ? row : M - m0 - 1;        // rows past the end are computed and dropped
        if (GROUPED && groups_rows) from = groups_rows[m0 + (int)from];
        a_at[i] = from * (uint32_t)(2 * K) + chunk * 16;
    }
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i) {
        const int row = (wave * W_LOADS + i) * LOAD_ROWS + lane / CHUNKS;
        const int chunk = (lane % CHUNKS) ^ chunk_swap<DEPTH>(row);
        const int of_part = MODE == MB_SWIGLU ? row - w_part * (BT / 2) : row;
        w_at[i] = (uint32_t)(of_part < N - n0 ? of_part : N - n0 - 1) * (uint32_t)(2 * K) + chunk * 16;
    }
    const fw_buffer a_rows = fw_make_buffer(a_base + k_first), w_rows = fw_make_buffer(w_base + k_first);
    // This wave's loads for a slab of either operand, into the stage at `stage`. A last slab of half the length has no upper
    // chunks: the lower ones are read again in their place and never used.
    const int whole = k_length / DEPTH, slabs = (k_length + DEPTH - 1) / DEPTH;
    auto request_a = [&](int stage, int slab, int i) { fw_buffer_to_lds(a_rows, lds + stage + (wave * A_LOADS + i) * 1024, a_at[i], slab * (DEPTH * 2)); };
    auto request_w = [&](int stage, int slab, int i) { fw_buffer_to_lds(w_rows, lds + stage + (wave * W_LOADS + i) * 1024, w_at[i], slab * (DEPTH * 2)); };
    auto upper = [&](int first_row) { return ((lane % CHUNKS) ^ chunk_swap<DEPTH>(first_row + lane / CHUNKS)) >= CHUNKS / 2; };
    auto request_slab_a = [&](int stage, int slab) {
#pragma unroll
        for (int i = 0; i < A_LOADS; ++i) {
            if (PARTS == 2 && slab >= whole && upper((wave * A_LOADS + i) * LOAD_ROWS)) a_at[i] -= BK * 2;
            request_a(stage, slab, i);
        }
    };
    auto request_slab_w = [&](int stage, int slab) {
#pragma unroll
        for (int i = 0; i < W_LOADS; ++i) {
            if (PARTS == 2 && slab >= whole && upper((wave * W_LOADS + i) * LOAD_ROWS)) w_at[i] -= BK * 2;
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
    // are 64 gate features (tiles 0 to 3) and the 64 up features of the same columns (tiles 4 to 7).
    // Every row this lane reads is (lane % 16) plus a multiple of 16: one permutation for all
    int slot[PARTS];
#pragma unroll
    for (int t = 0; t < PARTS; ++t) slot[t] = ((4 * t + (lane >> 4)) ^ chunk_swap<DEPTH>(lane & 15)) * 16;
    const int a_row0 = wm * (TM * 32) + (lane & 15), b_row0 = (MODE == MB_SWIGLU ? wn * 64 : wn * (TN * 32)) + (lane & 15);

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
            f.fa[which] = *reinterpret_cast<const bf16x8*>(lds + a_stage + slot[part] + (a_row0 + 16 * which) * (DEPTH * 2));
        } else {
            const int j = which - TA, row = MODE == MB_SWIGLU ? (j >> 2) * (BT / 2) + (j & 3) * 16 : j * 16;
            f.fb[j] = *reinterpret_cast<const bf16x8*>(lds + w_stage + slot[part] + (b_row0 + row) * (DEPTH * 2));
        }
    };
    auto read = [&](Operands& f, int a_stage, int w_stage, int part) {
#pragma unroll
        for (int u = 0; u < READS; ++u) read_one(f, a_stage, w_stage, part, u);
    };
    // product tile number `which`, row by row, every second row backwards
    auto multiply_one = [&](const Operands& f, int which) {
        const int i = which / TB, j = i & 1 ? TB - 1 - which % TB : which % TB;
        if constexpr (DEPTH == 32) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.fa[i], f.fb[j], acc[i][j], 0, 0, 0);
        else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(f.fa[i]), "v"(f.fb[j]));
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
    // that of a behind the MFMAs of the slab's last step, that of w behind those of the next slab's first (where a slab is one
    // step, both behind its later MFMAs).
    for (int u = 0; u < W_STAGES - 1; ++u) {
        if (u < slabs) request_slab_a(u * A_SLAB, u);
        if (u < slabs) request_slab_w(W_FIRST + u * W_SLAB, u);
    }
    if (A_STAGES == W_STAGES && A_STAGES <= slabs) request_slab_a((A_STAGES - 1) * A_SLAB, A_STAGES - 1);
    if (PARTS == 1 && W_STAGES <= slabs) request_slab_w(W_END - W_SLAB, W_STAGES - 1);
    if (slabs >= W_STAGES) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((A_STAGES - 1) * A_LOADS + (W_STAGES - (PARTS == 1 ? 1 : 2)) * W_LOADS) : "memory");
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
    if constexpr (PARTS == 2) {
        while (s + A_STAGES < whole) {
            arrived(f0);
#pragma unroll
            for (int u = 0; u < MFMAS; ++u) {
                if (u % READ_GAP == 0 && u / READ_GAP < READS) read_one(f1, a_now, w_now, 1, u / READ_GAP);
                if (u % W_GAP == 0 && u / W_GAP < W_LOADS) request_w(w_before, s + W_STAGES - 1, u / W_GAP);
                multiply_one(f0, u);
                __builtin_amdgcn_sched_barrier(0);
            }
            landed(f1);
#pragma unroll
            for (int u = 0; u < MFMAS; ++u) {
                if (u % READ_GAP == 0 && u / READ_GAP < READS) read_one(f0, a_then, w_then, 0, u / READ_GAP);
                if (u % A_GAP == 0 && u / A_GAP < A_LOADS) request_a(a_now, s + A_STAGES, u / A_GAP);
                multiply_one(f1, u);
                __builtin_amdgcn_sched_barrier(0);
            }
            advance();
            ++s;
        }
    } else {
        auto step = [&](const Operands& now, Operands& next) {
            landed(now);
#pragma unroll
            for (int u = 0; u < MFMAS; ++u) {
                if (u < READS) read_one(next, a_then, w_then, 0, u);
                const int load = (u - READS) / 2;
                if (u >= READS && (u - READS) % 2 == 0 && load < A_LOADS) request_a(a_now, s + A_STAGES, load);
                if (u >= READS && (u - READS) % 2 == 0 && load >= A_LOADS && load < SLAB_LOADS) request_w(w_now, s + W_STAGES, load - A_LOADS);
                multiply_one(now, u);
                __builtin_amdgcn_sched_barrier(0);
            }
            advance();
            ++s;
        };
        static_assert(PARTS == 2 || READS + 2 * SLAB_LOADS <= MFMAS, "the loads have MFMAs to go behind");
        while (s + A_STAGES + 1 < slabs) {                  // two slabs a turn, so that the operand sets keep their names
            step(f0, f1);
            step(f1, f0);
        }
    }
    // the last slabs: asking for what is left to ask for; one of two steps may have half the length
    for (; s < slabs; ++s) {
        const int ahead = (slabs < s + W_STAGES ? slabs : s + W_STAGES) - (s + 2);      // slabs behind s + 1 that have been asked for
        arrived(f0);
        if constexpr (PARTS == 2) {
            if (s < whole) read(f1, a_now, w_now, 1);
            if (s + W_STAGES - 1 < slabs) request_slab_w(w_before, s + W_STAGES - 1);
            multiply(f0);
            __builtin_amdgcn_sched_barrier(0);
            arrived(f1);
        }
        if (s + 1 < slabs) {
            wait_for_all_but(ahead);
            __builtin_amdgcn_s_barrier();
            read(PARTS == 2 ? f0 : f1, a_then, w_then, 0);
            if (s + A_STAGES < slabs) request_slab_a(a_now, s + A_STAGES);
            if (PARTS == 1 && s + W_STAGES < slabs) request_slab_w(w_now, s + W_STAGES);
        }
        if constexpr (PARTS == 2) {
            if (s < whole) multiply(f1);
        } else {
            multiply(f0);
            __builtin_amdgcn_sched_barrier(0);
            if (s + 1 < slabs) {
                arrived(f1);
                f0 = f1;
            }
        }
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
        f32x4 sum[TA][TB];
        for (int of = 0; of < cut.slices; ++of) {
            const fw_buffer theirs = left_by(of);
            f32x4 part[TA][TB];
#pragma unroll
            for (int u = 0; u < MFMAS; ++u) part[u / TB][u % TB] = fw_buffer_load_device(theirs, tid * 16, u * 4096);
#pragma unroll
            for (int u = 0; u < MFMAS; ++u) sum[u / TB][u % TB] = of ? sum[u / TB][u % TB] + part[u / TB][u % TB] : part[u / TB][u % TB];
        }
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
    const uint32_t first_row = (uint32_t)(wm * (TM * 32) + row_base);      // of this lane, of the tile
    // the eight rows of row tile i and pair j of column tiles that this lane holds: gated, or with the bias
    constexpr int PAIRS = MODE == MB_SWIGLU ? 2 : TN;
    auto values = [&](int i, int j, float b, float (&rows)[8]) {
        float left[4], right[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if constexpr (MODE == MB_SWIGLU) {
                left[r] = fw_gate_of<TO>(acc[i][2 * j][r], unit) * acc[i][2 * j + 4][r];
                right[r] = fw_gate_of<TO>(acc[i][2 * j + 1][r], unit) * acc[i][2 * j + 5][r];
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
    if (SIZE == 4 || ((N & 1) == 0 && (uintptr_t)out % 4 == 0)) {
#pragma unroll
        for (int j = 0; j < PAIRS; ++j) {
            const int c = (MODE == MB_SWIGLU ? wn * 64 : wn * (TN * 32)) + j * 32 + col;        // column of the tile
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
        return;
    }
    // Two bytes an element, and rows of an odd length or an output at an odd place: every element leaves by itself, just as free of branches
    // (with two an element 5,532 x 83 x 608 took 19.0 us against 11.5, 1,300 x 3,071 x 1,024 25.7 against 18.3).
    if constexpr (SIZE == 2) {
#pragma unroll
        for (int j = 0; j < PAIRS; ++j) {
            const int c = (MODE == MB_SWIGLU ? wn * 64 : wn * (TN * 32)) + j * 32 + col;
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
    }
}

template <int MODE, typename TO, int TN, int TM, int DEPTH, bool GROUPED, bool SPLIT = false>
static int launch_tiles(const void* a, const void* w, const float* bias, void* out, int M, int N, int K, int tiles_m, const BigGroups& groups,
                        hipStream_t stream, const BigSlices& cut = BigSlices()) {
    const int tiles_n = fw_ceil_div(N, MODE == MB_SWIGLU ? BT / 2 : BigTile<TM, TN, DEPTH>::WIDE);
    const int per_xcd = fw_ceil_div((long long)tiles_m * tiles_n * (SPLIT ? cut.slices : 1), 8);
    const int lds_bytes = BigTile<TM, TN, DEPTH>::LDS;
    static bool configured = false;     // per instantiation
    if (!configured) {
        hipError_t status = hipFuncSetAttribute((const void*)gemm_mfma_big_kernel<MODE, TO, TN, TM, DEPTH, GROUPED, SPLIT>,
                                                hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
        if (status != hipSuccess) {
            fw_set_error("gemm_mfma_big: cannot reserve %d bytes of LDS: %s", lds_bytes, hipGetErrorString(status));
            return -1;
        }
        configured = true;
    }
    gemm_mfma_big_kernel<MODE, TO, TN, TM, DEPTH, GROUPED, SPLIT><<<per_xcd * 8, 256, lds_bytes, stream>>>(
        (const uint16_t*)a, (const uint16_t*)w, bias, (TO*)out, M, N, K, tiles_m, tiles_n, per_xcd, N, groups, cut);
    return 0;
}
template <int MODE, typename TO, int TN = 4, int TM = 4>
static int launch_big(const void* a, const void* w, const float* bias, void* out, int M, int N, int K, hipStream_t stream) {
    return launch_tiles<MODE, TO, TN, TM, 64, false>(a, w, bias, out, M, N, K, fw_ceil_div(M, BigTile<TM, TN, 64>::ROWS), BigGroups(), stream);
}

// The grouped product of fw_grouped_gemm on tiles of 128 places by 256 rows of W, for K a multiple of 32 and a of less than 4 GB. Bound by
// the experts' weights from memory (600 MB for both products of 32 experts of 1,536 features: 127 us) and by tiles that an expert's last places fill partly.
// Slabs of 64 k leave room for one workgroup on a compute unit, slabs of 32 for two (three stages of 24 KB each), of which one multiplies while the other
// starts, ends or waits: a short K and experts of less than a tile of places, whose weights are the load, take the latter. us, slabs of 64 / 32, gated and
// down: 2,048 rows, 4 of 32 experts, 1,536 features over 2,048 146 / 147 and 90 / 99, 1,111 rows 108 / 115 and 49 / 53, 600 rows 109 / 105 and 37 / 37; 1,500
// rows, 2 of 8 over 4,096 97 / 110; 3,000 rows, 4 of 16 over 1,280 91 / 85; 2,048 rows, 2 of 8 over 1,024 57 / 52, 6 of 64 62 / 54. (On v_mfma_f32_32x32x16_bf16 with
// slabs of 32: 154 and 102, 120 and 57; tiles of 256 places 186; through registers, moe.hip, 241.)
bool fw_grouped_big_takes(int a_rows, int N, int K) { return K % BK == 0 && K <= BK_MOST && N <= BN_MOST && 2ll * a_rows * K <= 0xffff0000ll; }
int fw_launch_grouped_big(const void* a, const int32_t* place_row, const void* w, const int32_t* expert_begin, void* out, int gated, int places,
                          int experts, int N, int K, hipStream_t stream) {
    const BigGroups groups = {place_row, expert_begin, experts};
    const int tiles_m = places / 128 + (experts < places ? experts : places);       // at most: every expert's last tile may not be full
    // (what the product through registers, whose tiles have half the features, would refuse is refused here too)
    FW_REQUIRE((long long)tiles_m * fw_ceil_div(N, gated ? BT / 4 : BT / 2) < (1ll << 30), "grouped_gemm: too many tiles");
    if (K >= 1536 && places >= 128 * experts) {
        if (gated) return launch_tiles<MB_SWIGLU, bf16_t, 4, 2, 64, true>(a, w, nullptr, out, places, N, K, tiles_m, groups, stream);
        return launch_tiles<MB_STORE, float, 4, 2, 64, true>(a, w, nullptr, out, places, N, K, tiles_m, groups, stream);
    }
    if (gated) return launch_tiles<MB_SWIGLU, bf16_t, 4, 2, 32, true>(a, w, nullptr, out, places, N, K, tiles_m, groups, stream);
    return launch_tiles<MB_STORE, float, 4, 2, 32, true>(a, w, nullptr, out, places, N, K, tiles_m, groups, stream);
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

// ----- K cut into slices, for products with at most half as many tiles as compute units and a long K --------
// A tile of 128 x 256 moves 48 bytes a clock of full MFMA rate through a compute unit's memory path, one of 128 x 128 all of its 64: two or three slices of K on
// the larger tiles pay for their meeting (about 12 us: 128 KB a workgroup out past the dies' caches and back) where K is long. us, cut / 128 x 128 with
// K dealt to the waves: storing 1,111 x 2,048 x 8,192 49.6 / 60.3, adding 2,048 x 2,048 x 8,192 72.2 / 70.5 alone and 8 us less of it in a prompt's step
// (4,863 against 4,995 for 16 layers), storing 1,024 x 2,560 x 6,368 51.2 / 73 (whole large tiles). With four slices the sum at the end costs more than it
// gives (adding 801 x 2,048 x 7,168 40.6 against 38.7 on 128 x 64), and so do slices of less than 512 k (2,048 x 1,024 x 1,024 21.2 / 12.2).
struct BigSplitPlan {
    int tiles, slices, k_each;
    size_t workspace_bytes;
};
static BigSplitPlan big_split_plan(int M, int N, int K) {
    BigSplitPlan plan = {0, 0, 0, 0};
    const long long tiles = (long long)fw_ceil_div(M, BT / 2) * fw_ceil_div(N, BT);
    if (tiles > 128) return plan;
    int slices = (int)(256 / tiles);                    // at most a workgroup a compute unit
    slices = slices > 3 ? 3 : slices;                   // the last workgroup of a tile adds them one after the other
    const int most = K / 512;
    slices = slices > most ? most : slices;
    if (slices < 2) return plan;
    plan.tiles = (int)tiles;
    plan.k_each = fw_ceil_div(fw_ceil_div(K, slices), 64) * 64;
    plan.slices = fw_ceil_div(K, plan.k_each);
    plan.workspace_bytes = (size_t)plan.slices * plan.tiles * (BT / 2) * BT * sizeof(float);
    return plan;
}

// What fw_gemm_mfma_big_split needs for a shape: its slices of K (0: it does not take the shape), bytes of float32 workspace and the number of
// int32 counters (zero before the first call; left zero).
extern "C" int fw_gemm_mfma_big_split_plan(int mode, int M, int N, int K, int* slices, size_t* workspace_bytes, int* counters) {
    FW_REQUIRE(M >= 1 && N > 0 && K > 0 && mode >= 0 && mode <= 2, "gemm_mfma_big_split: M %d N %d K %d mode %d", M, N, K, mode);
    BigSplitPlan plan = {0, 0, 0, 0};
    if (mode != MB_SWIGLU && K % BK == 0 && K <= BK_MOST && N <= BN_MOST) plan = big_split_plan(M, N, K);
    *slices = plan.slices;
    *workspace_bytes = plan.workspace_bytes;
    *counters = plan.tiles;
    return 0;
}

// fw_gemm_mfma's contract for modes 0 and 1, with K cut into slices as fw_gemm_mfma_big_split_plan says, on tiles of 128 x 256. Calls that overlap on one
// device must not share counters or workspace.
extern "C" int fw_gemm_mfma_big_split(const void* a, const void* w, const float* bias, void* out, int out_dtype, int mode, int M, int N, int K,
                                      void* workspace, size_t workspace_bytes, int* counters, int counters_len, void* stream) {
    int slices = 0, need_counters = 0;
    size_t need_bytes = 0;
    if (fw_gemm_mfma_big_split_plan(mode, M, N, K, &slices, &need_bytes, &need_counters)) return -1;
    FW_REQUIRE(slices > 1, "gemm_mfma_big_split: this shape (M %d N %d K %d mode %d) is not cut", M, N, K, mode);
    FW_REQUIRE(mode != MB_ACCUMULATE || out_dtype == FW_F32, "gemm_mfma_big_split: accumulation needs a float32 destination");
    FW_REQUIRE(out_dtype == FW_F32 || out_dtype == FW_BF16 || (out_dtype == FW_BF16_GELU && mode == MB_STORE), "gemm_mfma_big_split: unknown out dtype %d", out_dtype);
    FW_REQUIRE(((uintptr_t)a % 16 == 0) && ((uintptr_t)w % 16 == 0), "gemm_mfma_big_split: operands must be 16-byte aligned");
    FW_REQUIRE(workspace != nullptr && workspace_bytes >= need_bytes && counters != nullptr && counters_len >= need_counters && (uintptr_t)workspace % 16 == 0,
               "gemm_mfma_big_split: this shape needs %zu bytes of workspace and %d counters", need_bytes, need_counters);
    const BigSplitPlan plan = big_split_plan(M, N, K);
    const BigSlices cut = {plan.slices, plan.k_each, (float*)workspace, counters};
    const int tiles_m = fw_ceil_div(M, BT / 2);
    hipStream_t s = (hipStream_t)stream;
    int status;
    if (mode == MB_ACCUMULATE) status = launch_tiles<MB_ACCUMULATE, float, 4, 2, 64, false, true>(a, w, bias, out, M, N, K, tiles_m, BigGroups(), s, cut);
    else if (out_dtype == FW_F32) status = launch_tiles<MB_STORE, float, 4, 2, 64, false, true>(a, w, bias, out, M, N, K, tiles_m, BigGroups(), s, cut);
    else if (out_dtype == FW_BF16_GELU) status = launch_tiles<MB_STORE, gelu_bf16_t, 4, 2, 64, false, true>(a, w, bias, out, M, N, K, tiles_m, BigGroups(), s, cut);
    else status = launch_tiles<MB_STORE, bf16_t, 4, 2, 64, false, true>(a, w, bias, out, M, N, K, tiles_m, BigGroups(), s, cut);
    if (status != 0) return status;
    FW_LAUNCH_CHECK("gemm_mfma_big_split");
    return 0;
}
