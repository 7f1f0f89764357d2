// Matrix product out[M][N] = a[M][K] . w[N][K]^T (+ bias) of float32 operands on the float32 matrix
// instruction (v_mfma_f32_16x16x4_f32: full products, float32 sums), for any number of rows.
//
// What bounds it: for a few rows the stream of W, for many the matrix cores' float32 rate (157 TFLOP/s).
// The plain FMA tiles this replaces gave a decode step's product with 1,024 outputs 16 workgroups that
// walked K in order.
//
//  * K is cut into sixteen parts. For a few tiles a workgroup has sixteen waves, a part each; otherwise four, which
//    walk four parts in turn. (Below 256 k a part is at most a group of 16: the four waves then take groups in turn, as the first of
//    four would otherwise have most of them.) Each wave computes the whole tile over its parts; the partial tiles meet in LDS. A
//    tile of 64 x 64 reads 8 KB a wave for 2,048 cycles of matrix work: L2 carries that easily.
//  * Operands go straight into LDS (global_load_lds_dwordx4), each wave's into a ring of its own, a few groups of 16 k
//    ahead, and from there into registers one group ahead: nothing is shared between waves before the end, so there
//    is no barrier in the loop. Four neighbouring lanes ask for 64 contiguous bytes. Loaded in the order in which the
//    instruction wants them, neighbouring lanes ask for different rows, and a load costs its compute unit 64 lookups
//    instead of 16: one row 13.0 -> 10.7 us, 64 rows 19.7 -> 13.0 us for 1,024 outputs, K 4,608.
//  * Tiles are 16, 32 or 64 rows by as many columns; the host takes the ones that load the busiest
//    compute unit least (see pick). 16-wide tiles give a product of 1,024 outputs 64 workgroups of sixteen
//    waves with eight kilobytes of W in flight each.
//  * Every output is the sum over the same groups of the same four k in the same order, part by part, the parts
//    four by four, whatever the tile: its value does not depend on M or on the other rows.
//
// One row over K from 1,024 to 8,192 goes to gemm_float32_few.hip, which gives the same bits, and so do two rows below 32,768 features, adding over K up to
// 4,096, storing and gated over K 1,024 (fw_gemm_float32_few_takes).
//
// Measured inside a request of the LFM2-350M shape in float32, before -> after: one row, 1,024 outputs (K 4,608 and 1,024
// in the mean) 464 -> 9.3 us, gate|up (2 x 4,608, K 1,024) 171 + 5 -> 13.6 us (2.8 TB/s of W), 65,536 outputs 255 -> 49 us (5.4
// TB/s); 301 rows, gate|up 222 + 5 -> 82 us (69 TFLOP/s), 1,024 outputs 523 -> 38 us; 2,048 rows by 1,024 outputs, K 4,608: 187 us
// (103 TFLOP/s). The sums' distance from 64 bits in that request's logits fell from 8.8e-6 to 2.4e-6.
#include "fw_common.h"
#include "fw_kernels.h"
#include "float32_few.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;

// A group of 16 k of 16 rows is 1 KB of LDS: row r at 64 r, its four pieces (of four k) permuted, piece p in place
// p ^ (r / 4 % 4), so that the reads of one piece of 16 rows cover all banks once. Instruction j of a group takes
// component j of every lane's piece, so its four k are j, 4 + j, 8 + j, 12 + j of the group.
template <int TM, int TN>
struct Operands {
    f32x4 a[TM], w[TN];
};
template <int TM, int TN>
__device__ __forceinline__ void multiply_group(const Operands<TM, TN>& f, f32x4 (&acc)[TM][TN]) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int n = 0; n < TN; ++n) acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.w[n][j], f.a[i][j], acc[i][n], 0, 0, 0);
}

// groups of a wave in LDS or on their way there
template <int TM, int TN, int WAVES>
struct Ring {
    static constexpr int LOADS = TM + TN;                               // of a group, 1 KB each
    static constexpr int STAGES = WAVES == 16 ? (LOADS == 2 ? 4 : 3) : LOADS == 8 ? 2 : LOADS == 6 ? 3 : LOADS == 5 ? 4 : LOADS == 4 ? 5 : LOADS == 3 ? 6 : 8;
    static constexpr int BYTES = STAGES * LOADS * 1024;
};

// SwiGLU: w holds N gate rows, then N up rows; column tiles alternate between 16 gate rows and the up rows of the same
// features, so that one thread meets both at the end.
template <int TM, int TN, int WAVES, int MODE, typename TO>
__device__ __forceinline__ void gemm_float32_tile(const float* __restrict__ a, const float* __restrict__ w, const float* __restrict__ bias,
                                                  TO* __restrict__ out, int M, int N, int K, int tiles_m, int tiles_n, int per_xcd, int quads) {
    constexpr int ROWS = TM * 16, WIDE = TN * 16;                       // of a tile, in rows of a and of w
    constexpr int FEATURES = MODE == MF_SWIGLU ? WIDE / 2 : WIDE;       // outputs of a tile's row
    constexpr int LOADS = Ring<TM, TN, WAVES>::LOADS, STAGES = Ring<TM, TN, WAVES>::STAGES;
    constexpr bool FOLDS = WAVES < PARTS;                               // a wave walks several parts
    __shared__ __attribute__((aligned(1024))) unsigned char lds[WAVES * Ring<TM, TN, WAVES>::BYTES];
    static_assert(sizeof(float) * WAVES * ROWS * WIDE <= sizeof(lds), "the partial tiles take the rings' place");
    // workgroups are dealt to the dies in turn: a die gets neighbouring tiles, all rows of a column of tiles in a row
    const int logical = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (logical >= tiles_m * tiles_n) return;
    const int m0 = logical % tiles_m * ROWS, n0 = logical / tiles_m * FEATURES;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = lane & 15, piece = lane >> 4;                       // of an operand and of a product
    const int ask_row = lane >> 2, ask_piece = (lane & 3) ^ ((lane >> 4) & 3);      // of a load: place l % 4 of row l / 4

    // rows past the end are computed from the last one and dropped
    const float* a_row[4];      // TM and TN of them are used (sized so, the host pass emits the launch stub)
    const float* w_row[4];
#pragma unroll
    for (int i = 0; i < TM; ++i) a_row[i] = a + (size_t)min(m0 + i * 16 + ask_row, M - 1) * K;
#pragma unroll
    for (int n = 0; n < TN; ++n) {
        const int feature = MODE == MF_SWIGLU ? min(n0 + (n >> 1) * 16 + ask_row, N - 1) + (n & 1) * N : min(n0 + n * 16 + ask_row, N - 1);
        w_row[n] = w + (size_t)feature * K;
    }
    f32x4 acc[TM][TN], total[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int n = 0; n < TN; ++n) acc[i][n] = total[i][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    const int part = (K + PARTS * 16 - 1) / (PARTS * 16);               // groups of 16 k in a part
    const bool in_turn = FOLDS && K < PARTS * 16;
    const int k_step = in_turn ? WAVES * 16 : 16, k_begin = in_turn ? wave * 16 : wave * (PARTS / WAVES) * part * 16;
    const int k_end = in_turn ? K : min(K, k_begin + (PARTS / WAVES) * part * 16);
    const int groups = k_end > k_begin ? (k_end - k_begin + k_step - 1) / k_step : 0;
    unsigned char* ring = lds + wave * Ring<TM, TN, WAVES>::BYTES;
    auto request = [&](int group) {
        unsigned char* stage = ring + group % STAGES * (LOADS * 1024);
        const int k = min(k_begin + group * k_step + ask_piece * 4, K - 4);     // pieces past the end of K are set to zero below
#pragma unroll
        for (int n = 0; n < TN; ++n)
            __builtin_amdgcn_global_load_lds(w_row[n] + k, reinterpret_cast<uint32_t*>(stage + n * 1024), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < TM; ++i)
            __builtin_amdgcn_global_load_lds(a_row[i] + k, reinterpret_cast<uint32_t*>(stage + (TN + i) * 1024), 16, 0, 0);
    };
    const int place = row * 64 + ((piece ^ ((row >> 2) & 3)) << 4);
    auto read = [&](Operands<TM, TN>& f, int group) {
        const unsigned char* stage = ring + group % STAGES * (LOADS * 1024) + place;
#pragma unroll
        for (int n = 0; n < TN; ++n) f.w[n] = *reinterpret_cast<const f32x4*>(stage + n * 1024);
#pragma unroll
        for (int i = 0; i < TM; ++i) f.a[i] = *reinterpret_cast<const f32x4*>(stage + (TN + i) * 1024);
    };
    // the operands have left LDS: their stage may be written again
    auto arrived = [&](const Operands<TM, TN>& f) {
#pragma unroll
        for (int n = 0; n < TN; ++n) asm volatile("" ::"v"(f.w[n]));
#pragma unroll
        for (int i = 0; i < TM; ++i) asm volatile("" ::"v"(f.a[i]));
    };
    auto wait_for_all_but = [&](int ahead) {                            // groups that may still be on their way
        if (ahead >= 7) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(7 * LOADS) : "memory");
        else if (ahead >= 5) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(5 * LOADS) : "memory");
        else if (ahead >= 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * LOADS) : "memory");
        else if (ahead == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LOADS) : "memory");
        else if (ahead == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };
    int left = part;                                                    // groups until the part ends
    auto multiply = [&](const Operands<TM, TN>& f) {
        multiply_group<TM, TN>(f, acc);
        if constexpr (FOLDS) {
            if (--left == 0) {
                fw_mfma_drain();
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int n = 0; n < TN; ++n) {
                        total[i][n] += acc[i][n];
                        acc[i][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                    }
                left = part;
            }
        }
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
            } else if (k_begin + g * k_step + piece * 4 >= K) {         // K is no multiple of 16
#pragma unroll
                for (int n = 0; n < TN; ++n) now.w[n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int i = 0; i < TM; ++i) now.a[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
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
    __syncthreads();                                                    // every wave has left its ring
    fw_mfma_drain();

    // Lane (row l % 16 of a) holds features 4 * (l / 16) + r of each 16 x 16 product. A row's runs of four features lie permuted,
    // run q in place q ^ r (the low bits), so that sixteen rows' runs are written to all banks.
    constexpr int RUNS = WIDE / 4, OUT_RUNS = FEATURES / 4, ITEMS = ROWS * OUT_RUNS, THREADS = WAVES * 64;
    constexpr int PER_THREAD = (ITEMS + THREADS - 1) / THREADS;         // runs of four outputs
    f32x4* partial = reinterpret_cast<f32x4*>(lds);                     // [WAVES][ROWS][RUNS]
    auto place_of = [&](int r, int run) { return r * RUNS + (run ^ (r & (RUNS - 1))); };
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int n = 0; n < TN; ++n)
            partial[wave * ROWS * RUNS + place_of(i * 16 + row, n * 4 + piece)] = FOLDS ? total[i][n] + acc[i][n] : acc[i][n];
    f32x4 old[PER_THREAD];
    if constexpr (MODE == MF_ACCUMULATE) {
#pragma unroll
        for (int u = 0; u < PER_THREAD; ++u) {
            const int item = tid + u * THREADS, m = m0 + item / OUT_RUNS, n = n0 + item % OUT_RUNS * 4;
            if (quads && item < ITEMS && m < M && n < N) old[u] = *reinterpret_cast<const f32x4*>(out + (size_t)m * N + n);
        }
    }
    fw_lds_barrier();

    auto sum = [&](int r, int run) {
        const f32x4* from = partial + place_of(r, run);
        f32x4 quarter[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            quarter[q] = from[q * (WAVES / 4) * ROWS * RUNS];
#pragma unroll
            for (int p = 1; p < WAVES / 4; ++p) quarter[q] += from[(q * (WAVES / 4) + p) * ROWS * RUNS];
        }
        return ((quarter[0] + quarter[1]) + quarter[2]) + quarter[3];
    };
#pragma unroll
    for (int u = 0; u < PER_THREAD; ++u) {
        const int item = tid + u * THREADS, r = item / OUT_RUNS, f = item % OUT_RUNS * 4;
        const int m = m0 + r, n = n0 + f;
        if (item >= ITEMS || m >= M || n >= N) continue;
        f32x4 v;
        if constexpr (MODE == MF_SWIGLU) {
            const int run = ((f >> 4) * 32 + (f & 15)) / 4;
            const f32x4 g = sum(r, run), up = sum(r, run + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = g[e] * sigmoid_float32(g[e]) * up[e];
        } else {
            v = sum(r, f / 4);
            if (bias)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] += n + e < N ? bias[n + e] : 0.0f;
        }
        TO* to = out + (size_t)m * N + n;
        if (quads) {
            if constexpr (MODE == MF_ACCUMULATE) v += old[u];
            if constexpr (sizeof(TO) == 4) {
                *reinterpret_cast<f32x4*>(to) = v;
            } else {
                uint2 packed;
                packed.x = (uint32_t)float_to_bf16_bits(v[0]) | ((uint32_t)float_to_bf16_bits(v[1]) << 16);
                packed.y = (uint32_t)float_to_bf16_bits(v[2]) | ((uint32_t)float_to_bf16_bits(v[3]) << 16);
                *reinterpret_cast<uint2*>(to) = packed;
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (n + e >= N) continue;
                if constexpr (MODE == MF_ACCUMULATE) v[e] += load_as_float(to, e);
                store_from_float(to, e, v[e]);
            }
        }
    }
}

template <int TM, int TN, int WAVES, int MODE, typename TO>
__global__ __launch_bounds__(WAVES * 64) void gemm_float32_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                                  const float* __restrict__ bias, TO* __restrict__ out, int M, int N,
                                                                  int K, int tiles_m, int tiles_n, int per_xcd, int quads) {
    gemm_float32_tile<TM, TN, WAVES, MODE, TO>(a, w, bias, out, M, N, K, tiles_m, tiles_n, per_xcd, quads);
}
// The same in 256 registers, two workgroups on a compute unit (a tile of 64 x 64 otherwise takes 356): for a short K, where a tile
// is mostly its start and its end. 8,192 outputs, K 64, 4,096 rows: 144 -> 83 us, 2,048 outputs 38 -> 24; from K 512 on two
// tiles beside each other get in each other's way (1,024 outputs, K 4,608, 2,048 rows: 186 -> 220; K 1,024, 2,048 outputs, 1,000
// rows: 50 -> 58).
template <int TM, int TN, int WAVES, int MODE, typename TO>
__global__ __launch_bounds__(WAVES * 64) __attribute__((amdgpu_waves_per_eu(2))) void gemm_float32_short_kernel(
    const float* __restrict__ a, const float* __restrict__ w, const float* __restrict__ bias, TO* __restrict__ out, int M, int N, int K,
    int tiles_m, int tiles_n, int per_xcd, int quads) {
    gemm_float32_tile<TM, TN, WAVES, MODE, TO>(a, w, bias, out, M, N, K, tiles_m, tiles_n, per_xcd, quads);
}

namespace {

constexpr int SHORT_K = 512;        // below it the form for a short K

// The tile that loads the busiest compute unit least. A wave's group of 16 k costs a compute unit the matrix time of
// TM x TN products (128 cycles each on its SIMD) or the reading of TM + TN operands by four waves (about as many cycles
// each), whichever is more; the larger tile at a tie. Sixteen waves where the tiles are too few to hide a wave's walk
// through a quarter of K (1,024 outputs, K 4,608, one row: 72 groups one after the other against 18). Counting fractions of a
// round instead of whole ones took narrower tiles for wide outputs and lost (9,216 outputs, one row: 14.4 -> 16.0 us).
void pick(int M, int features, int K, bool pairs, int* best_m, int* best_n, int* waves) {
    long long best = -1, best_tiles = 0;
    for (int tm = 4; tm >= 1; tm /= 2)
        for (int tn = 4; tn >= (pairs ? 2 : 1); tn /= 2) {
            if (tm > 1 && tm * 8 >= M) continue;                        // half of the tile's rows would be empty
            const long long tiles = (long long)fw_ceil_div(M, tm * 16) * fw_ceil_div(features, tn * (pairs ? 8 : 16));
            const long long cost = fw_ceil_div(tiles, 256) * (long long)(tm * tn > tm + tn ? tm * tn : tm + tn);
            if (best < 0 || cost < best) {
                best = cost;
                best_tiles = tiles;
                *best_m = tm;
                *best_n = tn;
            }
        }
    *waves = *best_m * *best_n <= 2 && best_tiles <= 512 && K >= 512 ? 16 : 4;
}

template <int TM, int TN, int WAVES, int MODE, typename TO>
void run(const float* a, const float* w, const float* bias, void* out, int M, int N, int K, hipStream_t stream) {
    const int tiles_m = fw_ceil_div(M, TM * 16), tiles_n = fw_ceil_div(N, MODE == MF_SWIGLU ? TN * 8 : TN * 16);
    const int per_xcd = fw_ceil_div((long long)tiles_m * tiles_n, 8);
    const int quads = N % 4 == 0 && (uintptr_t)out % 16 == 0;
    if constexpr (TM * TN == 16) {
        if (K < SHORT_K) {
            gemm_float32_short_kernel<TM, TN, WAVES, MODE, TO><<<per_xcd * 8, WAVES * 64, 0, stream>>>(a, w, bias, (TO*)out, M, N, K, tiles_m, tiles_n, per_xcd, quads);
            return;
        }
    }
    gemm_float32_kernel<TM, TN, WAVES, MODE, TO><<<per_xcd * 8, WAVES * 64, 0, stream>>>(a, w, bias, (TO*)out, M, N, K, tiles_m, tiles_n, per_xcd, quads);
}

template <int MODE, typename TO>
void choose(const float* a, const float* w, const float* bias, void* out, int M, int N, int K, hipStream_t stream) {
    int tm = 1, tn = 2, waves = 4;
    pick(M, N, K, MODE == MF_SWIGLU, &tm, &tn, &waves);
#define FW_TILE(TM_, TN_, WAVES_) \
    if (tm == TM_ && tn == TN_ && waves == WAVES_) return run<TM_, TN_, WAVES_, MODE, TO>(a, w, bias, out, M, N, K, stream)
    FW_TILE(4, 4, 4); FW_TILE(4, 2, 4); FW_TILE(2, 4, 4); FW_TILE(2, 2, 4); FW_TILE(1, 4, 4); FW_TILE(1, 2, 4); FW_TILE(1, 2, 16);
    if constexpr (MODE != MF_SWIGLU) {
        FW_TILE(4, 1, 4); FW_TILE(2, 1, 4); FW_TILE(2, 1, 16); FW_TILE(1, 1, 4); FW_TILE(1, 1, 16);
    }
#undef FW_TILE
}

}  // namespace

extern "C" int fw_gemm_float32(const float* a, const float* w, const float* bias, void* out, int out_dtype, int mode, int M, int N,
                               int K, void* stream) {
    FW_REQUIRE(M >= 0 && N > 0 && K > 0 && K % 4 == 0, "gemm_float32: bad sizes M=%d N=%d K=%d", M, N, K);
    FW_REQUIRE(mode >= 0 && mode <= 2, "gemm_float32: unknown mode %d", mode);
    FW_REQUIRE(out_dtype == FW_F32 || (out_dtype == FW_BF16 && mode == MF_STORE), "gemm_float32: output dtype %d in mode %d", out_dtype, mode);
    FW_REQUIRE(mode != MF_SWIGLU || !bias, "gemm_float32: SwiGLU takes no bias");
    FW_REQUIRE(((uintptr_t)a | (uintptr_t)w) % 16 == 0, "gemm_float32: operands must be aligned to 16 bytes");
    FW_REQUIRE((long long)fw_ceil_div(M, 16) * fw_ceil_div(N, 8) < (1ll << 30), "gemm_float32: M=%d N=%d are too many tiles", M, N);
    if (M == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    if (fw_gemm_float32_few_takes(M, N, K, mode, false)) return fw_launch_float32_few(a, nullptr, nullptr, 0.0f, 0, w, bias, out, out_dtype, mode, M, N, K, s);
    if (mode == MF_ACCUMULATE) choose<MF_ACCUMULATE, float>(a, w, bias, out, M, N, K, s);
    else if (mode == MF_SWIGLU) choose<MF_SWIGLU, float>(a, w, nullptr, out, M, N, K, s);
    else if (out_dtype == FW_F32) choose<MF_STORE, float>(a, w, bias, out, M, N, K, s);
    else choose<MF_STORE, bf16_t>(a, w, bias, out, M, N, K, s);
    FW_LAUNCH_CHECK("gemm_float32");
    return 0;
}
