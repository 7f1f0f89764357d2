// Matrix product for up to 64 rows and a very wide output (a vocabulary's head): out[M][N] = a[M][K] . w[N][K]^T, bfloat16
// operands, float32 accumulation on the matrix cores. Bound by reading W once from HBM; a (up to 1 MB) is read from L2 by
// every workgroup.
//
//  * a workgroup (4 waves) owns 64 consecutive features over all of K, 16 of them to a wave: with so many features every
//    compute unit has several workgroups, one's end beside another's loads;
//  * W goes from global memory straight into MFMA operand registers (lane (n, g) of the 16x16x32
//    instruction holds k = 8g..8g+7 of feature n), four chunks of 64 k in flight per wave;
//  * a is staged through LDS once per workgroup (two buffers, one barrier per chunk), also
//    four chunks ahead in registers, and read from there as MFMA operands by every wave.
//
// Every global load is unconditional (addresses clamped into the operands, a zeroed outside K on its way to LDS): a
// branch around a load, or arithmetic right behind it, makes the compiler wait for loads in flight. The barriers order
// LDS traffic only, for the same reason. 65,536 features over K 2,048 at 16 / 64 rows: 50.5 / 62 us; on the tiles of up to
// 64 x 64 of gemm_rows.hip, one workgroup to a compute unit, 52 / 70 us.
// The reference has no counterpart for this batch size: its decode projections are
// one-warp-per-row vector kernels run per request (native/include/flyweight_v2_qwen_kernels.hpp:855-941).
#include "fw_common.h"
#include "fw_kernels.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

#define GM_THREADS 256
#define GM_DEPTH 4      // chunks in flight
#define GM_PAD 8        // bfloat16 elements between LDS rows: spreads the rows over the banks

struct MediumArgs {
    const uint16_t* a;
    const uint16_t* w;
    const float* bias;
    void* out;
    int M, N, K;
    // prepared activations: a = x * w of an RMS norm, left by an accumulating product together with
    // these sums; the rows' 1/rms is formed here and applied to the sums of the product
    const float* squares;           // [squares_rows][row stride]
    int squares_rows;
    float eps;
    int rotate;                     // workgroups start their walk over K at different chunks
};

// rows of the sums of squares are 16 wide for up to 16 rows of a (the fused decode product's
// layout), 64 wide beyond
__host__ __device__ inline int gm_square_stride(int M) { return M <= 16 ? 16 : 64; }

// MT: tiles of 16 rows of a.
template <int MT, typename TO, bool ROTATE, bool WT>
__global__ __launch_bounds__(GM_THREADS) void gemm_medium_kernel(const MediumArgs p) {
    constexpr int CHUNK = 64;                   // k per iteration
    constexpr int SEG = CHUNK / 8;              // 16-byte pieces per row of a chunk of a
    constexpr int PIECES = MT * 16 * SEG;       // pieces per chunk of a
    constexpr int AP = (PIECES + GM_THREADS - 1) / GM_THREADS;
    constexpr int STRIDE = CHUNK + GM_PAD;
    __shared__ __attribute__((aligned(16))) uint16_t a_lds[2][MT * 16][STRIDE];
    __shared__ float square_parts[GM_THREADS], inv_rows[64];

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r16 = lane & 15, g = lane >> 4;
    const int M = p.M, N = p.N, K = p.K;
    const int square_stride = gm_square_stride(M);
    const int tile = blockIdx.x;
    const int n0 = tile * 64;
    const int chunks = (K + CHUNK - 1) / CHUNK;
    const int iterations = (chunks + GM_DEPTH - 1) / GM_DEPTH * GM_DEPTH;

    const int feature = n0 + 16 * wave + r16 < N ? n0 + 16 * wave + r16 : 0;
    const uint16_t* w_row = WT ? p.w + ((size_t)(feature >> 4) * (size_t)(K >> 5) << 9) + (((g << 4) | (feature & 15)) << 3)
                               : p.w + (size_t)feature * K;
    const uint16_t* a_piece[AP];
    int piece_row[AP], piece_k[AP];
#pragma unroll
    for (int i = 0; i < AP; ++i) {
        const int q = threadIdx.x + i * GM_THREADS;
        piece_row[i] = q / SEG;
        piece_k[i] = (q % SEG) * 8;
        a_piece[i] = p.a + (size_t)min(piece_row[i], M - 1) * K;
    }

    bf16x8 wf[GM_DEPTH][2], areg[GM_DEPTH][AP];
    f32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Nothing is done to a loaded value before the chunk is used (a select right behind a load
    // would wait for it at once): W comes from a clamped address as it is, and the rows of a are
    // zeroed outside the slice when they move to LDS, three chunks after their load.
    // Workgroups walk K from different chunks on (and around): all of them read the same rows of a, and in step they would
    // ask one cache line of it at a time from every compute unit at once. Where a workgroup starts depends on its tile
    // alone, so the order of its sum over K does not depend on the batch or on timing (inside a decode step of 8 rows the
    // head 59.8 -> 50.3 us).
    const int rotate = ROTATE ? (int)(tile * 5u % (unsigned)chunks) : 0;
    auto chunk_start = [&](const int c) {
        if (!ROTATE) return c * CHUNK;
        if (c >= chunks) return K;                      // past the end: nothing of it is inside
        const int turned = c + rotate;
        return (turned < chunks ? turned : turned - chunks) * CHUNK;
    };
    auto load = [&](const int d, const int c) {
        const int k0 = chunk_start(c);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int k = k0 + ks * 32 + g * 8;
            // (chunks begin at multiples of 32, and K is one where W lies in tiles: a tile's columns are inside or outside together)
            wf[d][ks] = fw_load_weights<WT>(w_row + (k < K ? (WT ? (size_t)(k >> 5) << 9 : (size_t)k) : 0));
        }
#pragma unroll
        for (int i = 0; i < AP; ++i) {
            const int k = k0 + piece_k[i];
            areg[d][i] = *reinterpret_cast<const bf16x8*>(a_piece[i] + (k < K ? k : 0));
        }
    };
    auto stage = [&](const int d, const int buffer, const int c) {
        const bf16x8 none = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < AP; ++i)
            if (PIECES % GM_THREADS == 0 || piece_row[i] < MT * 16) {
                // K is a multiple of 8: a run of 8 is inside or outside as a whole
                const bool inside = chunk_start(c) + piece_k[i] < K;
                *reinterpret_cast<bf16x8*>(&a_lds[buffer][piece_row[i]][piece_k[i]]) = inside ? areg[d][i] : none;
            }
    };
    auto multiply = [&](const int d, const int buffer) {
        bf16x8 af[2][MT];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                af[ks][mt] = *reinterpret_cast<const bf16x8*>(&a_lds[buffer][mt * 16 + r16][ks * 32 + g * 8]);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[d][ks], af[ks][mt], acc[mt], 0, 0, 0);
    };

    // prepared activations: this thread's share of the sums of squares of one row is asked for
    // first and added up behind the first chunks of W (a wave issues in order: a sum formed here
    // would hold the stream of W back by a round trip)
    constexpr int SQ_HELD = 32;
    float held[SQ_HELD];
    if (p.squares) {
        const int row = threadIdx.x % square_stride, part = threadIdx.x / square_stride, parts = GM_THREADS / square_stride;
        const float* from = p.squares + row;
        const int last = p.squares_rows - 1;
#pragma unroll
        for (int u = 0; u < SQ_HELD; ++u) {
            const int e = part + u * parts;
            held[u] = from[(size_t)(e < last ? e : last) * square_stride];
        }
    }
#pragma unroll
    for (int d = 0; d < GM_DEPTH; ++d) load(d, d);
    // the shares of the sums of squares have been on their way since before W: they are the
    // oldest loads, so adding them up here waits for nothing that was asked for after them
    float square_share = 0.0f;
    if (p.squares) {
        const int row = threadIdx.x % square_stride, part = threadIdx.x / square_stride, parts = GM_THREADS / square_stride;
        float share[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < SQ_HELD; ++u) share[u & 3] += part + u * parts < p.squares_rows ? held[u] : 0.0f;
        const float* from = p.squares + row;
        for (int e = part + SQ_HELD * parts; e < p.squares_rows; e += parts) share[0] += from[(size_t)e * square_stride];
        square_share = (share[0] + share[1]) + (share[2] + share[3]);
    }
    stage(0, 0, 0);
    if (p.squares) square_parts[threadIdx.x] = square_share;
    fw_lds_barrier();
    if (p.squares && threadIdx.x < square_stride) {
        // the shares of a row meet in a fixed order; read in the epilogue, many barriers from here
        float total = 0.0f;
        for (int part = 0; part < GM_THREADS / square_stride; ++part) total += square_parts[part * square_stride + threadIdx.x];
        inv_rows[threadIdx.x] = rsqrtf(total / (float)K + p.eps);
    }
    for (int c0 = 0; c0 < iterations; c0 += GM_DEPTH) {
#pragma unroll
        for (int d = 0; d < GM_DEPTH; ++d) {
            // chunk c0 + d: its W is in register set d, its a in LDS buffer d % 2; the next chunk's a
            // waits in register set d + 1 and moves to the other buffer; set d is then refilled
            multiply(d, d & 1);
            stage((d + 1) % GM_DEPTH, (d + 1) & 1, c0 + d + 1);
            load(d, c0 + d + GM_DEPTH);
            fw_lds_barrier();       // LDS only: the loads just issued stay in flight
        }
    }
    fw_mfma_drain();     // branches follow that lead to code reading the accumulators

    // D layout of the 16x16 product: lane holds features 4 * (lane / 16) + r of the wave's tile
    // for row lane % 16 of a
    const int n_first = n0 + 16 * wave + 4 * g;
    const bool whole = n_first + 3 < N && (N & 3) == 0;     // four features in one aligned piece
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = mt * 16 + r16;
        if (m >= M) continue;
        const size_t at = (size_t)m * N + n_first;
        float v[4];
        const float inv = p.squares ? inv_rows[m] : 1.0f;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = fw_before_store<TO>(acc[mt][r] * inv + ((p.bias && n_first + r < N) ? p.bias[n_first + r] : 0.0f));
        if constexpr (sizeof(TO) == 4) {
            float* to = reinterpret_cast<float*>(p.out) + at;
            if (whole) {
                *reinterpret_cast<f32x4*>(to) = f32x4{v[0], v[1], v[2], v[3]};
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (n_first + r < N) to[r] = v[r];
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
                for (int r = 0; r < 4; ++r)
                    if (n_first + r < N) to[r] = float_to_bf16_bits(v[r]);
            }
        }
    }
}

// ----- host side ---------------------------------------------------------------------------

template <int MT, bool ROTATE, bool WT>
static void medium_launch_as(const MediumArgs& args, int out_dtype, int tiles, hipStream_t stream) {
    if (out_dtype == FW_F32) gemm_medium_kernel<MT, float, ROTATE, WT><<<tiles, GM_THREADS, 0, stream>>>(args);
    else if (out_dtype == FW_BF16_GELU) gemm_medium_kernel<MT, gelu_bf16_t, ROTATE, WT><<<tiles, GM_THREADS, 0, stream>>>(args);
    else gemm_medium_kernel<MT, bf16_t, ROTATE, WT><<<tiles, GM_THREADS, 0, stream>>>(args);
}

template <int MT>
static void medium_launch(const MediumArgs& args, bool tiled, int out_dtype, int tiles, hipStream_t stream) {
    if (args.rotate) {
        if (tiled) medium_launch_as<MT, true, true>(args, out_dtype, tiles, stream);
        else medium_launch_as<MT, true, false>(args, out_dtype, tiles, stream);
    } else {
        if (tiled) medium_launch_as<MT, false, true>(args, out_dtype, tiles, stream);
        else medium_launch_as<MT, false, false>(args, out_dtype, tiles, stream);
    }
}

extern "C" int fw_gemm_medium(const void* a, const void* w, int w_tiled, const float* bias, void* out, int out_dtype, int M, int N, int K,
                              const float* squares, int squares_rows, float eps, void* stream) {
    FW_REQUIRE(M >= 1 && M <= 64, "gemm_medium: takes 1..64 rows, got %d", M);
    FW_REQUIRE(N > 0 && K > 0 && K % 8 == 0, "gemm_medium: K (%d) must be a positive multiple of 8, N (%d) positive", K, N);
    FW_REQUIRE(!w_tiled || K % 32 == 0, "gemm_medium: weights in operand tiles need K (%d) to be a multiple of 32", K);
    FW_REQUIRE(out_dtype == FW_F32 || out_dtype == FW_BF16 || out_dtype == FW_BF16_GELU, "gemm_medium: unknown out dtype %d", out_dtype);
    FW_REQUIRE(((uintptr_t)a | (uintptr_t)w | (uintptr_t)out) % 16 == 0, "gemm_medium: operands must be 16-byte aligned");
    FW_REQUIRE(squares == nullptr || (squares_rows >= 1 && eps > 0.0f), "gemm_medium: prepared activations come with their sums of squares and eps");
    const int tiles = fw_ceil_div(N, 64);
    FW_REQUIRE(tiles <= 65535 * 16, "gemm_medium: too many tiles");
    MediumArgs args;
    args.a = (const uint16_t*)a; args.w = (const uint16_t*)w; args.bias = bias; args.out = out;
    args.M = M; args.N = N; args.K = K;
    args.squares = squares; args.squares_rows = squares_rows; args.eps = eps;
    args.rotate = (long long)N * K > (1ll << 24);
    hipStream_t s = (hipStream_t)stream;
    if (M <= 16) medium_launch<1>(args, w_tiled != 0, out_dtype, tiles, s);
    else if (M <= 32) medium_launch<2>(args, w_tiled != 0, out_dtype, tiles, s);
    else medium_launch<4>(args, w_tiled != 0, out_dtype, tiles, s);
    FW_LAUNCH_CHECK("gemm_medium");
    return 0;
}
