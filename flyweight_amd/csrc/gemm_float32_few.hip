// Matrix product of one or two rows, float32: out[M][N] = a[M][K] . w[N][K]^T, optionally with the rows' RMS norm in front. The float32 matrix
// instruction (gemm_float32.hip) computes sixteen rows whether they are there or not, and a tile of sixteen features gives a product of 1,024
// outputs 64 workgroups: a fourth of the chip streams W, through 4 us of matrix time. Here every output is formed by ordinary multiply-adds in the order
// of that instruction (its four k one after the other, each a fused multiply-add: bit for bit the same on normal and subnormal numbers), so
// that a value does not depend on the kernel that formed it:
//
//  * a workgroup has 4 or 16 rows of W and all of K, which is cut into sixteen parts: wave q has parts 4 q .. 4 q + 3, a lane one row of W and one part.
//    With 16 rows of W a lane takes the rows of a in turn; with 4 a wave has four places for rows of a, of which two at most are filled and the others form
//    the first row's sums once more. A lane walks its part in groups of 16 k; the parts meet in LDS at the end and are added as there;
//  * W goes straight into LDS, each wave's into a ring of its own up to sixteen groups deep (64 KB a workgroup in flight), 64 contiguous bytes a row of W
//    and part; no barrier in the loop;
//  * the rows of a lie in LDS, normed on the way there. They are asked for ahead of W, so that nothing waits for W before it is needed; the norm's
//    chain (load, sum over the workgroup, scale) runs while W is on its way and the kernel that did it alone is saved.
//
// Bound by the stream of W (1,024 x 4,608: 2.3 TB/s, 4,608 gated x 1,024 3.1, 65,536 x 1,024 5.4) and by the kernel's start and end. Four rows of W a workgroup below
// 3,072 outputs, 16 from there on and for gated products (3,072 storing 5.7 with 16, 6.3 with 4; 2,048 5.1 and 4.8).
#include "fw_common.h"
#include "fw_kernels.h"
#include "float32_few.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;

#define FEW_WIDE 3072                   // outputs from which a workgroup has 16 rows of W
#define FEW_ROWS 2
#define FEW_HOLD 8                      // runs of four floats of the rows that a thread holds on their way to LDS
#define NORM_RUNS 4                     // of one row with a norm: K up to 4,096

// A workgroup barrier that orders LDS traffic alone. (fw_lds_barrier waits for loads to LDS as well, here for all of W that is on its way.)
__device__ __forceinline__ void meet() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// part: groups of 16 k in a part of K; STAGES groups of a wave are in LDS or on their way there (at most `part`: the first ones are asked for
// without a condition, so that the rows' arrival is told from theirs)
template <int F, int STAGES, int MODE, typename TO, bool NORM>
__global__ __launch_bounds__(256) void gemm_float32_few_kernel(const float* __restrict__ a, const float* __restrict__ norm_weight,
                                                               const int32_t* __restrict__ row_index, float eps, int one_centered,
                                                               const float* __restrict__ w, const float* __restrict__ bias, TO* __restrict__ out, int M, int N,
                                                               int K, int part) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];       // [rings of the four waves][rows of a, part by part]
    constexpr int LOADS = F / 4, RING = STAGES * LOADS * 1024;       // loads of 1 KB of a group
    constexpr int FEATURES = MODE == MF_SWIGLU ? F / 2 : F;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = blockIdx.x * FEATURES;
    const int part_bytes = part * 64 + 16, row_bytes = PARTS * part_bytes;       // of a row of a in LDS (a part starts in other banks than the one before)
    unsigned char* ring = lds + wave * RING;
    unsigned char* rows = lds + 4 * RING;
    __shared__ float scratch[FEW_ROWS][4];

    // the rows
    f32x4 held[FEW_HOLD];
    f32x4 scale[NORM ? NORM_RUNS : 1];
    const int runs = K / 4;
    if constexpr (NORM) {
#pragma unroll
        for (int m = 0; m < FEW_ROWS; ++m) {
            const int of = m < M ? m : 0;
            const f32x4* source = reinterpret_cast<const f32x4*>(a + (size_t)(row_index ? row_index[of] : of) * K);
#pragma unroll
            for (int u = 0; u < NORM_RUNS; ++u) {
                const int run = tid + u * 256;
                held[m * NORM_RUNS + u] = source[run < runs ? run : 0];
            }
        }
#pragma unroll
        for (int u = 0; u < NORM_RUNS; ++u) scale[u] = reinterpret_cast<const f32x4*>(norm_weight)[tid + u * 256 < runs ? tid + u * 256 : 0];
    } else {
#pragma unroll
        for (int u = 0; u < FEW_HOLD; ++u) {
            const int run = tid + u * 256;                  // (a condition around a load would wait for it)
            held[u] = reinterpret_cast<const f32x4*>(a)[run < M * runs ? run : 0];
        }
    }
    // the old values that this thread's output adds to
    const int item_row = tid / FEATURES, item = tid % FEATURES;
    const bool mine = item_row < M && n0 + item < N;
    float old = 0.0f;
    if (MODE == MF_ACCUMULATE) old = load_as_float(out, mine ? (size_t)item_row * N + n0 + item : 0);
    __builtin_amdgcn_sched_barrier(0);

    // W: load number `i` of a group brings 16 runs of 64 bytes, run r a row of W and part (F 16: row r, part i; F 4: row r % 4, part r / 4); its pieces
    // of 16 bytes are stored permuted, piece p in place p ^ (r / 4 % 4)
    const int ask = lane >> 2, ask_piece = (lane & 3) ^ ((ask >> 2) & 3);
    const int ask_row = F == 16 ? ask : ask & 3, ask_part = F == 16 ? 0 : ask >> 2;
    int feature = n0 + (MODE == MF_SWIGLU ? ask_row & 7 : ask_row);
    feature = feature < N ? feature : N - 1;            // rows past the end are computed from the last one and dropped
    const uint32_t row_at = (uint32_t)(feature - n0 + (MODE == MF_SWIGLU && ask_row >= 8 ? N : 0)) * (uint32_t)(K * 4);
    // (the address is the same in every lane, which the compiler has to be told: it would load lane by lane)
    const uint64_t at = (uint64_t)(w + (size_t)n0 * K);
    const uint32_t low = __builtin_amdgcn_readfirstlane((uint32_t)at), high = __builtin_amdgcn_readfirstlane((uint32_t)(at >> 32));
    const fw_buffer rows_of_w = fw_make_buffer(reinterpret_cast<const void*>((uint64_t)high << 32 | low));
    auto request = [&](int group) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int k = (wave * 4 + (F == 16 ? i : ask_part)) * part * 16 + group * 16 + ask_piece * 4;       // (past the end of K: not counted below)
            fw_buffer_to_lds(rows_of_w, ring + (group % STAGES) * (LOADS * 1024) + i * 1024, row_at + (uint32_t)(k < K ? k : K - 4) * 4, 0);
        }
    };
#pragma unroll
    for (int s = 0; s < STAGES; ++s) request(s);
    __builtin_amdgcn_sched_barrier(0);

    auto place = [&](int m, int run) { return reinterpret_cast<f32x4*>(rows + m * row_bytes + (run / (part * 4)) * part_bytes + (run % (part * 4)) * 16); };
    if constexpr (NORM) {
        const float one = one_centered ? 1.0f : 0.0f;
        float inv[FEW_ROWS];
#pragma unroll
        for (int m = 0; m < FEW_ROWS; ++m) {
            if (m >= M) break;
            float sum = 0.0f;
#pragma unroll
            for (int u = 0; u < NORM_RUNS; ++u) {
                const f32x4 v = tid + u * 256 < runs ? held[m * NORM_RUNS + u] : f32x4{0.f, 0.f, 0.f, 0.f};
                sum += fw_sum_of_squares(v);
            }
            sum = wave_sum(sum);
            if (lane == 0) scratch[m][wave] = sum;
        }
        meet();
#pragma unroll
        for (int m = 0; m < FEW_ROWS; ++m) {
            if (m >= M) break;
            inv[m] = rsqrtf((((scratch[m][0] + scratch[m][1]) + scratch[m][2]) + scratch[m][3]) / (float)K + eps);
        }
#pragma unroll
        for (int m = 0; m < FEW_ROWS; ++m) {
            if (m >= M) break;
#pragma unroll
            for (int u = 0; u < NORM_RUNS; ++u) {
                const int run = tid + u * 256;
                if (run >= runs) break;
                f32x4 y;
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] = held[m * NORM_RUNS + u][e] * inv[m] * (scale[u][e] + one);
                *place(m, run) = y;
            }
        }
    } else {
#pragma unroll
        for (int u = 0; u < FEW_HOLD; ++u) {
            const int run = tid + u * 256;
            if (run < M * runs) *place(run / runs, run % runs) = held[u];
        }
    }
    meet();

    // a lane's row of W, part, and row of a (F 16: all of them in turn)
    const int run16 = lane & 15, my_part = F == 16 ? lane >> 4 : (lane >> 2) & 3, slot = lane >> 4;
    const int my_row = F == 16 ? 0 : (slot < M ? slot : 0);
    const unsigned char* w_at = ring + (F == 16 ? my_part * 1024 : 0) + run16 * 64;
    const unsigned char* a_at = rows + my_row * row_bytes + (wave * 4 + my_part) * part_bytes;
    const int swap = (run16 >> 2) & 3, k_first = (wave * 4 + my_part) * part * 16;
    const bool ragged = K % (PARTS * 16) != 0;
    constexpr int SUMS = F == 16 ? FEW_ROWS : 1;
    float acc[SUMS] = {};
    struct Operands {
        f32x4 x[4], y[SUMS][4];
    };
    auto read = [&](Operands& f, int group) {
        const unsigned char* stage = w_at + (group % STAGES) * (LOADS * 1024);
#pragma unroll
        for (int i = 0; i < 4; ++i) f.x[i] = *reinterpret_cast<const f32x4*>(stage + (i ^ swap) * 16);
#pragma unroll
        for (int m = 0; m < SUMS; ++m)
            if (m == 0 || m < M)
#pragma unroll
                for (int i = 0; i < 4; ++i) f.y[m][i] = *reinterpret_cast<const f32x4*>(a_at + m * row_bytes + group * 64 + i * 16);
    };
    // the operands have left LDS: their stage may be written again
    auto arrived = [&](const Operands& f) { asm volatile("" ::"v"(f.x[0]), "v"(f.x[1]), "v"(f.x[2]), "v"(f.x[3]) : "memory"); };
    auto multiply = [&](Operands& f, int group) {
        if (ragged)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (k_first + group * 16 + i * 4 >= K) {
                    f.x[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int m = 0; m < SUMS; ++m) f.y[m][i] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
#pragma unroll
        for (int m = 0; m < SUMS; ++m)
            if (m == 0 || m < M)
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[m] = fmaf(f.x[i][j], f.y[m][i][j], acc[m]);
    };
    // while a group is multiplied the next one is read from LDS and those behind it are on their way
    Operands even, odd;
    int g = 0;
    auto steady = [&](Operands& now, Operands& next) {
        arrived(now);
        request(g + STAGES);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 1) * LOADS) : "memory");
        read(next, g + 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(now, g);
        ++g;
    };
    auto last = [&](Operands& now, Operands& next) {
        arrived(now);
        if (g + 1 < part) {
            const int left = (part - 2 - g) * LOADS;        // loads behind the next group's
            if (left >= 12) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
            else if (left >= 8) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
            else if (left >= 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
            else if (left == 3) asm volatile("s_waitcnt vmcnt(3)" ::: "memory");
            else if (left == 2) asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
            else if (left == 1) asm volatile("s_waitcnt vmcnt(1)" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            read(next, g + 1);
        }
        multiply(now, g);
        ++g;
    };
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 1) * LOADS) : "memory");
    read(even, 0);
    while (g + STAGES + 1 < part) {
        steady(even, odd);
        steady(odd, even);
    }
    if (g + STAGES < part) {
        steady(even, odd);
        even = odd;
    }
    while (g < part) {
        last(even, odd);
        if (g < part) last(odd, even);
    }

    // the parts meet: [part][row of a][row of W]
    __syncthreads();
    float* partial = reinterpret_cast<float*>(lds);
    if constexpr (F == 16) {
#pragma unroll
        for (int m = 0; m < FEW_ROWS; ++m)
            if (m < M) partial[((wave * 4 + my_part) * FEW_ROWS + m) * F + run16] = acc[m];
    } else {
        if (slot < FEW_ROWS) partial[((wave * 4 + my_part) * FEW_ROWS + slot) * F + (lane & 3)] = acc[0];
    }
    __syncthreads();
    if (!mine) return;
    auto sum = [&](int f) {
        const float* from = partial + item_row * F + f;
        float quarter[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            quarter[q] = from[q * 4 * FEW_ROWS * F];
#pragma unroll
            for (int p = 1; p < 4; ++p) quarter[q] += from[(q * 4 + p) * FEW_ROWS * F];
        }
        return ((quarter[0] + quarter[1]) + quarter[2]) + quarter[3];
    };
    float v;
    if constexpr (MODE == MF_SWIGLU) {
        const float gate = sum(item), up = sum(item + F / 2);
        v = gate * sigmoid_float32(gate) * up;
    } else {
        v = sum(item);
        if (bias) v += bias[n0 + item];
    }
    if (MODE == MF_ACCUMULATE) v += old;
    store_from_float(out, (size_t)item_row * N + n0 + item, v);
}

namespace {

template <int F, int STAGES, int MODE, typename TO, bool NORM>
int run(const float* a, const float* norm_weight, const int32_t* row_index, float eps, int one_centered, const float* w, const float* bias, void* out, int M,
        int N, int K, hipStream_t stream) {
    const int part = fw_ceil_div(K, PARTS * 16);
    const int bytes = STAGES * F * 1024 + M * PARTS * (part * 64 + 16);
    static bool configured = false;
    if (!configured) {
        hipError_t status = hipFuncSetAttribute((const void*)gemm_float32_few_kernel<F, STAGES, MODE, TO, NORM>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - 1024);
        FW_REQUIRE(status == hipSuccess, "gemm_float32: cannot reserve LDS: %s", hipGetErrorString(status));
        configured = true;
    }
    gemm_float32_few_kernel<F, STAGES, MODE, TO, NORM><<<fw_ceil_div(N, MODE == MF_SWIGLU ? F / 2 : F), 256, bytes, stream>>>(a, norm_weight, row_index, eps, one_centered, w,
                                                                                                       bias, (TO*)out, M, N, K, part);
    FW_LAUNCH_CHECK("gemm_float32");
    return 0;
}

template <int MODE, typename TO>
int choose(const float* a, const float* norm_weight, const int32_t* row_index, float eps, int one_centered, const float* w, const float* bias, void* out, int M,
           int N, int K, hipStream_t s) {
    if constexpr (MODE != MF_SWIGLU) {
        if (N < FEW_WIDE) {
            if (norm_weight) return run<4, 4, MODE, TO, true>(a, norm_weight, row_index, eps, one_centered, w, bias, out, M, N, K, s);
            if (K >= 16 * 256) return run<4, 16, MODE, TO, false>(a, norm_weight, row_index, eps, one_centered, w, bias, out, M, N, K, s);
            return run<4, 4, MODE, TO, false>(a, norm_weight, row_index, eps, one_centered, w, bias, out, M, N, K, s);
        }
    }
    if (norm_weight) return run<16, 4, MODE, TO, true>(a, norm_weight, row_index, eps, one_centered, w, bias, out, M, N, K, s);
    return run<16, 4, MODE, TO, false>(a, norm_weight, row_index, eps, one_centered, w, bias, out, M, N, K, s);
}

}  // namespace

// Whether a product of `M` rows goes here: a part of K has at least four groups (the first ones are asked for without a condition; below K 512 gemm_float32
// deals K out in another order), and rows that the threads hold. us, gemm_float32 / here (with the norm in front: as two kernels / here), one row: adding
// 1,024 x 4,608 13.3 / 8.2, 1,024 x 1,024 5.3 / 3.7, 2,048 x 8,192 24.6 / 19.5, gated 4,608 x 1,024 (16.8 / 12.4), 8,192 x 2,048 (30.9 / 26.8), storing 3,072 x 1,024
// (7.9 / 5.7), 65,536 x 1,024 (53.2 / 50.3). Two rows: adding 2,048 x 2,048 7.3 / 5.8, gated 4,608 x 1,024 (18.0 / 13.1), but storing 6,144 x 2,048 14.5 /
// 15.3 and 65,536 x 1,024 (53.6 / 53.7); four rows, gated 4,608 x 1,024 (18.5 / 23.3): a lane's multiply-adds are in line.
bool fw_gemm_float32_few_takes(int M, int N, int K, int mode, bool normed) {
    return M >= 1 && M <= FEW_ROWS && !(M == 2 && mode != MF_ACCUMULATE && K > 1024) && K % 4 == 0 && K >= 1024 && (long long)M * K <= FEW_HOLD * 1024 && (!normed || K <= NORM_RUNS * 1024) &&
           (long long)N * K * (mode == MF_SWIGLU ? 2 : 1) < (1ll << 29) && (M == 1 || N < 32768);
}

int fw_launch_float32_few(const float* a, const float* norm_weight, const int32_t* row_index, float eps, int one_centered, const float* w, const float* bias,
                          void* out, int out_dtype, int mode, int M, int N, int K, hipStream_t s) {
    if (mode == MF_ACCUMULATE) return choose<MF_ACCUMULATE, float>(a, norm_weight, row_index, eps, one_centered, w, bias, out, M, N, K, s);
    if (mode == MF_SWIGLU) return choose<MF_SWIGLU, float>(a, norm_weight, row_index, eps, one_centered, w, nullptr, out, M, N, K, s);
    if (out_dtype == FW_F32) return choose<MF_STORE, float>(a, norm_weight, row_index, eps, one_centered, w, bias, out, M, N, K, s);
    return choose<MF_STORE, bf16_t>(a, norm_weight, row_index, eps, one_centered, w, bias, out, M, N, K, s);
}

// fw_gemm_float32 over rows that pass an RMS norm first, as fw_rmsnorm_rows gives it bit for bit; fw_gemm_float32_normed_takes says for which shapes.
// fw_gemm_float32_few_rows: whether fw_gemm_float32 itself comes here.
extern "C" int fw_gemm_float32_few_rows(int mode, int M, int N, int K) { return fw_gemm_float32_few_takes(M, N, K, mode, false) ? 1 : 0; }
extern "C" int fw_gemm_float32_normed_takes(int mode, int M, int N, int K) { return fw_gemm_float32_few_takes(M, N, K, mode, true) ? 1 : 0; }
extern "C" int fw_gemm_float32_normed(const float* x, const float* norm_weight, const int32_t* row_index, float eps, int one_centered, const float* w,
                                      const float* bias, float* out, int mode, int M, int N, int K, void* stream) {
    FW_REQUIRE(mode == MF_STORE || mode == MF_SWIGLU, "gemm_float32_normed: mode %d", mode);
    FW_REQUIRE(M >= 1 && N > 0 && K > 0 && fw_gemm_float32_few_takes(M, N, K, mode, true), "gemm_float32_normed: M=%d N=%d K=%d are not taken", M, N, K);
    FW_REQUIRE(mode != MF_SWIGLU || !bias, "gemm_float32_normed: SwiGLU takes no bias");
    FW_REQUIRE(norm_weight && ((uintptr_t)x | (uintptr_t)w | (uintptr_t)norm_weight) % 16 == 0, "gemm_float32_normed: operands must be aligned to 16 bytes");
    return fw_launch_float32_few(x, norm_weight, row_index, eps, one_centered, w, bias, out, FW_F32, mode, M, N, K, (hipStream_t)stream);
}
