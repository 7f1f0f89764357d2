// Matrix product for a few dozen to a few hundred rows: out[M][N] = a[M][K] . w[N][K]^T, bfloat16 operands, float32
// accumulation on the matrix cores (decode steps of 17 requests and more, short prompts).
//
// What bounds it: the stream of W from memory and, as soon as there are more than a few rows, the bytes that each compute
// unit has to bring in (its tile's rows of a and of W; 64 bytes a clock at best), not the products. So the tile is chosen
// to give every compute unit the fewest rows to bring in, and nothing else stands in the way of the loads:
//
//  * A workgroup owns a tile of 16 to 64 rows by 16 to 64 rows of W over all of K; its waves take the groups of 64 k in
//    turn and each computes the whole tile over its own. Nothing is exchanged between workgroups.
//  * Operands go straight into LDS (global_load_lds_dwordx4), each wave's into a ring of its own, and from there into
//    registers one group of 64 k ahead. Waves share nothing before the end, so the loop has no barrier; a wave waits
//    for its own loads alone, counted. Eight neighbouring lanes ask for the 128 bytes of a row that are a line of L2: asked
//    for 64 at a time, with every compute unit at it, rows come in at 42-66 KB/us a compute unit instead of 85-120 (and at
//    37 in the order of the matrix operands, sixteen rows at neighbouring lanes).
//  * The partial tiles meet in LDS and are added in the order of the waves: the order of a sum depends on K and on the number of
//    waves, which the tile decides (M, N and the mode choose it), not on the other rows or on timing. (Eight parts of K whatever
//    the tile, the waves of a tile of four walking two each in sums of their own, would take M out of it; the tiles of four waves
//    were 3 to 8 % slower so, and four waves for the small tiles 10 to 25 %.)
//
// Measured against the product that cut K over workgroups, which met through a workspace and a ticket (every weight from
// memory; 64 rows, us): adding 2,048 features over K 8,192 / 2,048 17.7 -> 15.8 / 11.7 -> 7.0, 1,024 over 4,608 / 1,024 13.6 -> 8.4 /
// 7.9 -> 4.2, storing 6,144 / 3,072 over 2,048 12.3 -> 11.1 / 11.9 -> 8.5, gate|up 16,384 over 2,048 19.8 -> 18.8. With the shares of the
// sums of squares asked for behind the loop instead of ahead of it a product of prepared activations took 4-5 us more.
//
// Epilogues as in the other products: store (float32, bfloat16, gelu), add into the float32 residual stream (optionally
// leaving what the next norm needs), the gated unit.
#include "fw_common.h"
#include "fw_kernels.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

enum { GR_STORE = 0, GR_ACCUMULATE = 1, GR_GATED = 2 };

struct RowsArgs {
    const uint16_t* a;
    const uint16_t* w;
    const float* bias;
    void* out;
    int M, N, K;                    // N: output features (gated: w has 2N rows, gate then up)
    int tiles_m, tiles_n, per_xcd;
    int quads;                      // every row of out starts at 16 bytes
    // accumulating product: what the norm after it will need (all null: nothing)
    const float* next_norm_weight;  // [N]
    int next_one_centered;
    uint16_t* next_activations;     // bfloat16 [M][N] = x_new * (w_next or 1 + w_next)
    float* next_squares;            // [tiles_n][row stride]: the tile's sum of x_new^2 per row
    // prepared activations: a = x * w of an RMS norm, left by an accumulating product together with these sums; the rows'
    // 1/rms is formed here and applied to the sums of the product
    const float* squares;           // [squares_rows][row stride]
    int squares_rows;
    float eps;
    // the gated unit: limit 0: silu(gate) * up; < 0: gelu_tanh(gate) * up; else clamped halves (fw_gated_unit)
    float glu_limit, glu_alpha, glu_shift;
};

// rows of the sums of squares are 16 wide for up to 16 rows of a (the fused decode product's layout), 64 wide beyond
__host__ __device__ inline int gr_square_stride(int M) { return M <= 16 ? 16 : 64; }

__device__ __forceinline__ float gr_silu(float g) {
    if (g >= 0.0f) return g / (1.0f + __expf(-g));
    const float e = __expf(g);
    return g * e / (1.0f + e);
}

// eight waves, or four where a wave's group is large
constexpr int waves_of(int loads) { return loads <= 3 ? 8 : 4; }

// Groups of 64 k of a wave in LDS or on their way there: up to 144 of a compute unit's 160 KB, one workgroup on it.
template <int TM, int TN>
struct Ring {
    static constexpr int LOADS = 2 * (TM + TN);                 // of a group, 1 KB each
    static constexpr int WAVES = waves_of(TM + TN);
    static constexpr int STAGES = 144 / (WAVES * LOADS) > 8 ? 8 : 144 / (WAVES * LOADS);
    static constexpr int BYTES = STAGES * LOADS * 1024;         // of a wave
};

template <int TM, int TN>
struct Operands {
    bf16x8 a[2][TM], w[2][TN];                                  // of the group's two steps of 32 k
};

// A group's 16 rows of a are 2 KB of LDS: row r at 128 r, its eight pieces (of eight k) permuted, piece p in place
// p ^ (r / 2 % 8), so that the reads of one piece of 16 rows cover all banks once. Operand tiles of W (WT) already lie in the
// order in which the lanes want them, two of them side by side.
template <int TM, int TN, int MODE, typename TO, bool WT>
__global__ __launch_bounds__(waves_of(TM + TN) * 64) void gemm_rows_kernel(const RowsArgs p) {
    constexpr int WAVES = Ring<TM, TN>::WAVES, LOADS = Ring<TM, TN>::LOADS, STAGES = Ring<TM, TN>::STAGES, THREADS = WAVES * 64;
    constexpr int ROWS = TM * 16, WIDE = TN * 16;                       // of a tile, in rows of a and of w
    constexpr int FEATURES = MODE == GR_GATED ? WIDE / 2 : WIDE;        // outputs of a tile's row
    constexpr int QUADS = FEATURES / 4, ITEMS = ROWS * QUADS;           // four neighbouring outputs of a row
    constexpr int PER_THREAD = (ITEMS + THREADS - 1) / THREADS;
    constexpr int HELD = 128 * ROWS / THREADS;                          // shares of (128 rows of) the sums of squares asked for ahead
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    __shared__ float square_parts[THREADS], inv_rows[64];
    // workgroups are dealt to the dies in turn: a die gets neighbouring tiles, all rows of a column of tiles in a row
    const int logical = (blockIdx.x & 7) * p.per_xcd + (blockIdx.x >> 3);
    if (logical >= p.tiles_m * p.tiles_n) return;
    const int M = p.M, N = p.N, K = p.K;
    const int tile_m = logical % p.tiles_m, tile_n = logical / p.tiles_m;
    const int m0 = tile_m * ROWS, n0 = tile_n * FEATURES;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = lane & 15, piece = lane >> 4;                               // of an operand and of a product
    // of a load of rows: place l % 8 of row l / 8 (and of row 8 + l / 8 of the sixteen in the second load)
    const int ask_row = lane >> 3, ask_piece[2] = {(lane & 7) ^ (ask_row >> 1), (lane & 7) ^ (4 + (ask_row >> 1))};

    // What the epilogue reads beside the sums travels ahead of everything else: the residual's old values and the next norm's
    // weight for this thread's outputs, its share of the sums of squares.
    f32x4 old[PER_THREAD], next_weight[PER_THREAD];
    const bool quads = p.quads;
#pragma unroll
    for (int u = 0; u < PER_THREAD; ++u) {
        const int item = tid + u * THREADS, m = m0 + item / QUADS, n = n0 + item % QUADS * 4;
        const bool there = item < ITEMS && m < M && n + 3 < N && quads;
        if (MODE == GR_ACCUMULATE && quads) {
            old[u] = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(p.out) + (there ? (size_t)m * N + n : 0));
            if (p.next_activations) next_weight[u] = *reinterpret_cast<const f32x4*>(p.next_norm_weight + (there ? n : 0));
        }
    }
    const int square_stride = gr_square_stride(M);
    float held[HELD];
    if (p.squares)
#pragma unroll
        for (int u = 0; u < HELD; ++u) {
            const int e = tid / ROWS + u * (THREADS / ROWS);
            held[u] = p.squares[(size_t)(e < p.squares_rows ? e : 0) * square_stride + min(m0 + tid % ROWS, square_stride - 1)];
        }

    // rows past the end are computed from the last one and dropped
    const uint16_t* a_row[8];       // 2 TM and TN or 2 TN of them are used (sized so, the host pass emits the launch stub)
    const uint16_t* w_row[8];
#pragma unroll
    for (int i = 0; i < 2 * TM; ++i) a_row[i] = p.a + (size_t)min(m0 + i * 8 + ask_row, M - 1) * K;
    if constexpr (WT) {
#pragma unroll
        for (int n = 0; n < TN; ++n) {
            const int feature = min((MODE == GR_GATED ? n0 + (n >> 1) * 16 : n0 + n * 16) + row, N - 1) + (MODE == GR_GATED ? (n & 1) * N : 0);
            w_row[n] = p.w + ((size_t)(feature >> 4) * (size_t)(K >> 5) << 9) + (((piece << 4) | (feature & 15)) << 3);
        }
    } else {
#pragma unroll
        for (int n = 0; n < 2 * TN; ++n) {
            const int of = (MODE == GR_GATED ? n0 + (n >> 2) * 16 : n0 + (n >> 1) * 16) + (n & 1) * 8 + ask_row;
            w_row[n] = p.w + (size_t)(min(of, N - 1) + (MODE == GR_GATED ? (n >> 1 & 1) * N : 0)) * K;
        }
    }
    // the groups of 64 k go to the waves in turn; a short K goes to as many waves as have two of them each
    const int all_groups = (K + 63) / 64, walkers = min(WAVES, max(2, (all_groups + 1) / 2));
    const int groups = wave < walkers ? (all_groups - wave + walkers - 1) / walkers : 0;
    unsigned char* ring = lds + wave * Ring<TM, TN>::BYTES;
    const bool once = p.tiles_m == 1;                                   // nobody else reads this W
    auto request = [&](int group) {
        unsigned char* stage = ring + group % STAGES * (LOADS * 1024);
        const int k0 = (wave + group * walkers) * 64;
        const int k[2] = {min(k0 + ask_piece[0] * 8, K - 8), min(k0 + ask_piece[1] * 8, K - 8)};    // pieces past K are set to zero below
        if constexpr (WT) {
            const int second = k0 + 32 < K ? 512 : 0;                   // (K may end behind the first of the two tiles)
#pragma unroll
            for (int n = 0; n < TN; ++n)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const uint16_t* from = w_row[n] + (size_t)k0 * 16 + t * second;
                    uint32_t* to = reinterpret_cast<uint32_t*>(stage + (2 * n + t) * 1024);
                    if (once) __builtin_amdgcn_global_load_lds(from, to, 16, 0, 2);
                    else __builtin_amdgcn_global_load_lds(from, to, 16, 0, 0);
                }
        } else {
#pragma unroll
            for (int n = 0; n < 2 * TN; ++n)
                __builtin_amdgcn_global_load_lds(w_row[n] + k[n & 1], reinterpret_cast<uint32_t*>(stage + n * 1024), 16, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 2 * TM; ++i)
            __builtin_amdgcn_global_load_lds(a_row[i] + k[i & 1], reinterpret_cast<uint32_t*>(stage + (2 * TN + i) * 1024), 16, 0, 0);
    };
    const int place[2] = {row * 128 + ((piece ^ (row >> 1)) << 4), row * 128 + (((4 + piece) ^ (row >> 1)) << 4)};
    auto read = [&](Operands<TM, TN>& f, int group) {
        const unsigned char* stage = ring + group % STAGES * (LOADS * 1024);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
            for (int n = 0; n < TN; ++n)
                f.w[t][n] = *reinterpret_cast<const bf16x8*>(stage + n * 2048 + (WT ? t * 1024 + lane * 16 : place[t]));
#pragma unroll
            for (int i = 0; i < TM; ++i) f.a[t][i] = *reinterpret_cast<const bf16x8*>(stage + (TN + i) * 2048 + place[t]);
        }
    };
    // the operands have left LDS: their stage may be written again
    auto arrived = [&](const Operands<TM, TN>& f) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
            for (int n = 0; n < TN; ++n) asm volatile("" ::"v"(f.w[t][n]));
#pragma unroll
            for (int i = 0; i < TM; ++i) asm volatile("" ::"v"(f.a[t][i]));
        }
    };
    auto wait_for_all_but = [&](int ahead) {                            // groups that may still be on their way
        if (ahead >= 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * LOADS) : "memory");
        else if (ahead == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LOADS) : "memory");
        else if (ahead == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };
    f32x4 acc[TN][TM];
#pragma unroll
    for (int n = 0; n < TN; ++n)
#pragma unroll
        for (int i = 0; i < TM; ++i) acc[n][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto multiply = [&](const Operands<TM, TN>& f) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int n = 0; n < TN; ++n)
#pragma unroll
                for (int i = 0; i < TM; ++i) acc[n][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[t][n], f.a[t][i], acc[n][i], 0, 0, 0);
    };
    if (groups > 0) {
        Operands<TM, TN> even, odd;
        int g = 0;
        // while a group is multiplied the next one is read from LDS and those behind it are on their way
        auto steady = [&](const Operands<TM, TN>& now, Operands<TM, TN>& next) {
            arrived(now);
            request(g + STAGES);
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 1) * LOADS) : "memory");
            read(next, g + 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply(now);
            ++g;
        };
        auto last = [&](Operands<TM, TN>& now, Operands<TM, TN>& next) {
            arrived(now);
            if (g + STAGES < groups) request(g + STAGES);
            if (g + 1 < groups) {
                wait_for_all_but(min(groups, g + 1 + STAGES) - 2 - g);
                read(next, g + 1);
            }
#pragma unroll
            for (int t = 0; t < 2; ++t)
                if ((wave + g * walkers) * 64 + t * 32 + piece * 8 >= K) {       // K is no multiple of 64
                    const bf16x8 nothing = __builtin_bit_cast(bf16x8, f32x4{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
                    for (int n = 0; n < TN; ++n) now.w[t][n] = nothing;
#pragma unroll
                    for (int i = 0; i < TM; ++i) now.a[t][i] = nothing;
                }
            multiply(now);
            ++g;
        };
        for (int s = 0; s < STAGES && s < groups; ++s) request(s);
        wait_for_all_but(min(groups, STAGES) - 1);
        read(even, 0);
        while (g + STAGES + 1 < groups) {
            steady(even, odd);
            steady(odd, even);
        }
        while (g < groups) {
            last(even, odd);
            if (g < groups) last(odd, even);
        }
    }
    fw_mfma_drain();
    if (p.squares) {
        float share = 0.0f;
#pragma unroll
        for (int u = 0; u < HELD; ++u) share += tid / ROWS + u * (THREADS / ROWS) < p.squares_rows ? held[u] : 0.0f;
        for (int e = tid / ROWS + HELD * (THREADS / ROWS); e < p.squares_rows; e += THREADS / ROWS)
            share += p.squares[(size_t)e * square_stride + min(m0 + tid % ROWS, square_stride - 1)];
        square_parts[tid] = share;
    }
    __syncthreads();                                                    // every wave has left its ring
    // lane (row l % 16 of a) holds features 4 * (l / 16) + r of each 16 x 16 product
    float* partial = reinterpret_cast<float*>(lds);                     // [WAVES][ROWS][WIDE]
#pragma unroll
    for (int n = 0; n < TN; ++n)
#pragma unroll
        for (int i = 0; i < TM; ++i)
            *reinterpret_cast<f32x4*>(partial + ((size_t)wave * ROWS + i * 16 + row) * WIDE + n * 16 + piece * 4) = acc[n][i];
    if (p.squares && tid < ROWS) {
        float total = 0.0f;                                             // the shares of a row meet in a fixed order
        for (int part_of = 0; part_of < THREADS / ROWS; ++part_of) total += square_parts[part_of * ROWS + tid];
        inv_rows[tid] = rsqrtf(total / (float)K + p.eps);
    }
    fw_lds_barrier();

    auto sum = [&](int r, int column) {
        const float* from = partial + r * WIDE + column;
        f32x4 total = *reinterpret_cast<const f32x4*>(from);
#pragma unroll
        for (int v = 1; v < WAVES; ++v) total += *reinterpret_cast<const f32x4*>(from + v * ROWS * WIDE);
        return total;
    };
#pragma unroll
    for (int u = 0; u < PER_THREAD; ++u) {
        const int item = tid + u * THREADS;
        if (item >= ITEMS) continue;                                    // (whole waves: ITEMS is a multiple of 64)
        const int r = item / QUADS, f = item % QUADS * 4;
        const int m = m0 + r, n = n0 + f;
        const bool mine = m < M, whole = n + 3 < N && quads;
        const float inv = p.squares ? inv_rows[r] : 1.0f;
        f32x4 v;
        if (MODE == GR_GATED) {
            const int column = (f >> 4) * 32 + (f & 15);
            const f32x4 gate = sum(r, column), up = sum(r, column + 16);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                v[e] = fw_gated_unit(gate[e] * inv, up[e] * inv, p.glu_limit, p.glu_alpha, p.glu_shift, [](float g) { return gr_silu(g); });
        } else {
            v = sum(r, f);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = fw_before_store<TO>(v[e] * inv + ((p.bias && n + e < N) ? p.bias[n + e] : 0.0f));
        }
        const size_t at = (size_t)(mine ? m : 0) * N + n;
        if (mine) {
            if constexpr (sizeof(TO) == 4) {
                float* to = reinterpret_cast<float*>(p.out) + at;
                if (whole) {
                    if (MODE == GR_ACCUMULATE) v += old[u];
                    *reinterpret_cast<f32x4*>(to) = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (n + e >= N) continue;
                        if (MODE == GR_ACCUMULATE) v[e] += to[e];
                        to[e] = v[e];
                    }
                }
            } else {
                uint16_t* to = reinterpret_cast<uint16_t*>(p.out) + at;
                if (whole) {
                    uint2 packed;
                    packed.x = (uint32_t)float_to_bf16_bits(v[0]) | ((uint32_t)float_to_bf16_bits(v[1]) << 16);
                    packed.y = (uint32_t)float_to_bf16_bits(v[2]) | ((uint32_t)float_to_bf16_bits(v[3]) << 16);
                    *reinterpret_cast<uint2*>(to) = packed;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (n + e < N) to[e] = float_to_bf16_bits(v[e]);
                }
            }
        }
        // what the norm after this addition needs: x * w of that norm in bfloat16, and the tile's sum of x^2 per row; the
        // product that follows forms the row's 1/rms from those sums
        if (MODE == GR_ACCUMULATE && p.next_activations) {
            float square = 0.0f;
            if (mine) {
                const float one = p.next_one_centered ? 1.0f : 0.0f;
                if (whole) {
                    uint2 packed;
                    const f32x4 w = next_weight[u];
                    packed.x = (uint32_t)float_to_bf16_bits(v[0] * (w[0] + one)) | ((uint32_t)float_to_bf16_bits(v[1] * (w[1] + one)) << 16);
                    packed.y = (uint32_t)float_to_bf16_bits(v[2] * (w[2] + one)) | ((uint32_t)float_to_bf16_bits(v[3] * (w[3] + one)) << 16);
                    *reinterpret_cast<uint2*>(p.next_activations + at) = packed;
                    square = (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (n + e >= N) continue;
                        p.next_activations[at + e] = float_to_bf16_bits(v[e] * (p.next_norm_weight[n + e] + one));
                        square += v[e] * v[e];
                    }
                }
            }
#pragma unroll
            for (int offset = 1; offset < QUADS; offset *= 2) square += __shfl_xor(square, offset, 64);
            if (item % QUADS == 0 && m < square_stride) p.next_squares[(size_t)tile_n * square_stride + m] = square;
        }
    }
}

// ----- host side ---------------------------------------------------------------------------
namespace {

struct RowsPlan {
    int tm, tn, tiles_m, tiles_n;
};

// The tile that gives the busiest compute unit the fewest rows to bring in; the taller one at a tie (W is then read
// from memory by fewer workgroups).
RowsPlan rows_plan(int M, int N, int mode) {
    RowsPlan best = {};
    long long least = -1;
    for (int tm = 4; tm >= 1; tm /= 2)
        for (int tn = 4; tn >= (mode == GR_GATED ? 2 : 1); tn /= 2) {
            if (tm > 1 && tm * 8 >= M) continue;                        // half of the tile's rows would be empty
            const int tiles_m = fw_ceil_div(M, tm * 16), tiles_n = fw_ceil_div(N, tn * (mode == GR_GATED ? 8 : 16));
            const long long cost = fw_ceil_div((long long)tiles_m * tiles_n, 256) * (long long)(tm + tn);
            if (least < 0 || cost < least) {
                least = cost;
                best = {tm, tn, tiles_m, tiles_n};
            }
        }
    return best;
}

template <int TM, int TN, int MODE, typename TO, bool WT>
int rows_run(const RowsArgs& args, hipStream_t stream) {
    constexpr int bytes = Ring<TM, TN>::WAVES * Ring<TM, TN>::BYTES;
    static_assert(bytes >= (int)sizeof(float) * Ring<TM, TN>::WAVES * TM * TN * 256, "the partial tiles take the rings' place");
    static bool configured = false;     // per instantiation
    if (!configured) {
        hipError_t status = hipFuncSetAttribute((const void*)gemm_rows_kernel<TM, TN, MODE, TO, WT>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        FW_REQUIRE(status == hipSuccess, "gemm_rows: cannot reserve %d bytes of LDS: %s", bytes, hipGetErrorString(status));
        configured = true;
    }
    gemm_rows_kernel<TM, TN, MODE, TO, WT><<<args.per_xcd * 8, Ring<TM, TN>::WAVES * 64, bytes, stream>>>(args);
    return 0;
}

template <int MODE, typename TO, bool WT>
int rows_tile(const RowsArgs& args, const RowsPlan& plan, hipStream_t stream) {
#define FW_TILE(TM, TN) \
    if (plan.tm == TM && plan.tn == TN) return rows_run<TM, TN, MODE, TO, WT>(args, stream)
    FW_TILE(4, 4); FW_TILE(4, 2); FW_TILE(2, 4); FW_TILE(2, 2); FW_TILE(1, 4); FW_TILE(1, 2);
    if constexpr (MODE != GR_GATED) {
        FW_TILE(4, 1); FW_TILE(2, 1); FW_TILE(1, 1);
    }
#undef FW_TILE
    FW_REQUIRE(false, "gemm_rows: no tile of %d x %d", plan.tm, plan.tn);
    return -1;
}

template <bool WT>
int rows_mode(const RowsArgs& args, const RowsPlan& plan, int out_dtype, int mode, hipStream_t stream) {
    if (mode == GR_GATED) return rows_tile<GR_GATED, bf16_t, WT>(args, plan, stream);
    if (mode == GR_ACCUMULATE) return rows_tile<GR_ACCUMULATE, float, WT>(args, plan, stream);
    if (out_dtype == FW_F32) return rows_tile<GR_STORE, float, WT>(args, plan, stream);
    if (out_dtype == FW_BF16_GELU) return rows_tile<GR_STORE, gelu_bf16_t, WT>(args, plan, stream);
    return rows_tile<GR_STORE, bf16_t, WT>(args, plan, stream);
}

}  // namespace

// how many rows the sums of squares left for the next norm take (the second extent: 16 for M <= 16, else 64)
extern "C" int fw_gemm_rows_square_tiles(int M, int N) { return rows_plan(M, N, GR_ACCUMULATE).tiles_n; }

// Whether the tiles are one round over the compute units, and serve better than the products that tile both operands. With a long K
// those have caught up with the large tiles unless their own leave much of a round empty, which these do not where 200 to 240 (up
// to K 8,192 more) of them are wanted. us, here / there, storing 2,560 features at 128 rows over K 4,096 / 8,192 15.1 / 18.2,
// 28.2 / 25.5, at 160 rows over 8,192 26.0 / 32.8; gated 1,536 at 192 rows over 4,096 / 8,192 22.7 / 23.7, 39.2 / 33.4, at 320 rows over
// 8,192 37.9 / 58.1; gated 4,096 at 128 rows over 8,192 / 10,752 40.9 / 45.9, 61.9 / 53.9. (Storing, the tiles of 64 x 64 win at any K.)
extern "C" int fw_gemm_rows_round_fits(int mode, int M, int N, int K) {
    const RowsPlan plan = rows_plan(M, N, mode);
    const long long tiles = (long long)plan.tiles_m * plan.tiles_n;
    if (M < 1 || M > 4096 || tiles > 256) return 0;
    const int products = plan.tm * plan.tn;
    if (mode == GR_ACCUMULATE || products < 8 || (tiles >= 200 && (K <= 8192 || tiles <= 240))) return 1;
    if (products == 8) return K < 8192 || M <= 96;
    return mode == GR_STORE || K <= 5120;
}

extern "C" int fw_gemm_rows(const void* a, const void* w, int w_tiled, const float* bias, void* out, int out_dtype, int mode, int M, int N,
                            int K, const float* next_norm_weight, int next_one_centered, void* next_activations, float* next_squares,
                            const float* squares, int squares_rows, float eps, float glu_limit, float glu_alpha, float glu_shift, void* stream) {
    FW_REQUIRE(M >= 1 && M <= 4096, "gemm_rows: takes 1..4096 rows, got %d", M);
    FW_REQUIRE(N > 0 && K > 0 && K % 8 == 0, "gemm_rows: K (%d) must be a positive multiple of 8, N (%d) positive", K, N);
    FW_REQUIRE(mode >= 0 && mode <= 2, "gemm_rows: unknown mode %d", mode);
    FW_REQUIRE(!w_tiled || K % 32 == 0, "gemm_rows: weights in operand tiles need K (%d) to be a multiple of 32", K);
    FW_REQUIRE(mode != GR_ACCUMULATE || out_dtype == FW_F32, "gemm_rows: accumulation needs a float32 destination");
    FW_REQUIRE(mode != GR_GATED || (out_dtype == FW_BF16 && bias == nullptr), "gemm_rows: the gated unit stores bfloat16 and takes no bias");
    FW_REQUIRE(out_dtype == FW_F32 || out_dtype == FW_BF16 || (out_dtype == FW_BF16_GELU && mode == GR_STORE), "gemm_rows: unknown out dtype %d", out_dtype);
    FW_REQUIRE(((uintptr_t)a | (uintptr_t)w) % 16 == 0, "gemm_rows: operands must be 16-byte aligned");
    FW_REQUIRE((next_activations == nullptr) == (next_squares == nullptr) && (next_activations == nullptr) == (next_norm_weight == nullptr),
               "gemm_rows: the next norm's weight, activations and sums of squares come together");
    FW_REQUIRE(next_activations == nullptr || (mode == GR_ACCUMULATE && M <= 64), "gemm_rows: only the accumulating product of up to 64 rows prepares the next norm");
    FW_REQUIRE(squares == nullptr || (squares_rows >= 1 && eps > 0.0f && M <= 64), "gemm_rows: prepared activations (up to 64 rows) come with their sums of squares and eps");
    FW_REQUIRE(next_norm_weight == nullptr || ((uintptr_t)next_norm_weight % 16 == 0 && (uintptr_t)next_activations % 16 == 0) || N % 4 != 0,
               "gemm_rows: the next norm's weight and activations must be 16-byte aligned");
    const RowsPlan plan = rows_plan(M, N, mode);
    RowsArgs args;
    args.a = (const uint16_t*)a; args.w = (const uint16_t*)w; args.bias = bias; args.out = out;
    args.M = M; args.N = N; args.K = K;
    args.tiles_m = plan.tiles_m; args.tiles_n = plan.tiles_n; args.per_xcd = fw_ceil_div((long long)plan.tiles_m * plan.tiles_n, 8);
    args.quads = N % 4 == 0 && (uintptr_t)out % 16 == 0;
    args.next_norm_weight = next_norm_weight; args.next_one_centered = next_one_centered;
    args.next_activations = (uint16_t*)next_activations; args.next_squares = next_squares;
    args.squares = squares; args.squares_rows = squares_rows; args.eps = eps;
    args.glu_limit = glu_limit; args.glu_alpha = glu_alpha; args.glu_shift = glu_shift;
    const int status = w_tiled ? rows_mode<true>(args, plan, out_dtype, mode, (hipStream_t)stream)
                               : rows_mode<false>(args, plan, out_dtype, mode, (hipStream_t)stream);
    if (status != 0) return status;
    FW_LAUNCH_CHECK("gemm_rows");
    return 0;
}
