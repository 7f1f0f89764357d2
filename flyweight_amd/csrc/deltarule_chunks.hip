// The gated delta rule over prompts, sixteen tokens at a time on the float32 matrix instruction.
//
// Per head, with state S [dim][vdim], a token brings q, k (dim channels, unit vectors), v (vdim channels), a write strength
// beta and a decay g per key channel:   S <- diag(g) S;   u = beta (v - S^T k);   S <- S + k u^T;   o = S^T q.
// Walked token by token, a column's two sums over the key channels and the write between them are one dependent chain
// (0.14 to 0.21 us a token, whatever the width of the chip). Over a chunk of sixteen tokens with the state S0 ahead of it and
// G_i the product of the chunk's decays up to token i, the writes u_i solve a triangular system
//     u_i = beta_i (v_i - (G_i k_i)^T S0 - sum_{j < i} L_ij u_j),     L_ij = sum_c k_i[c] k_j[c] g_{j+1}[c] .. g_i[c],
// which is linear in S0: u = Uv - W S0 and o = Ov + Qe S0, and the state behind the chunk is
//     S = diag(G_15) S0 + sum_j (k_j g_{j+1} .. g_15) u_j^T.
// W, Qe [16][dim], Uv, Ov [16][vdim] and the written keys depend on no state: delta_chunk_kernel forms them for all chunks
// side by side (with the short convolutions, unit vectors and decays in front of them), and delta_walk_kernel is left with three
// products of 16 tokens a chunk. Decays only ever multiply from a token to a later one, each product formed as it is needed: no quotient of two
// products, nothing that a strong decay could drive to infinity. Everything is float32 (exact products, float32 sums).
//
// 16 heads of 128 channels (8 of q and k), one prompt of 1,111 rows, before -> after: what the recurrence reads 41 us and the walk 227 us
// (32 lanes a column) -> the chunks 43 us and the walk 68 us; 277 rows 13 + 61 -> 20 + 20 us. The distance from 64 bits did not grow
// (read-outs 2.03e-7 -> 2.02e-7, states 3.82e-7 -> 3.78e-7).
#include "deltarule.h"
#include "fw_kernels.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;

#define CHUNK 16

static __host__ __device__ __forceinline__ int delta_key_width(int dim) { return (dim + 63) & ~63; }
static __host__ __device__ __forceinline__ int delta_value_width(int vdim) { return (vdim + 15) & ~15; }

// What the walk reads of a chunk and head (the packet), D = dim rounded up to 64, V = vdim rounded up to 16, floats:
//   W [D / 16][16 tokens][16 channels] | Qe likewise | written keys [D][16 tokens] | G_15 [D] | Uv [V][16 tokens] | Ov likewise
extern "C" int fw_delta_packet_floats(int dim, int vdim) { return 49 * delta_key_width(dim) + 32 * delta_value_width(vdim); }

// Chunks of a step: those of segment s begin at chunk seg_row0[s] / 16 + s, which leaves every segment room for its own.
extern "C" int fw_delta_chunk_slots(int rows, int segments) { return rows / CHUNK + segments; }

// log(1 + e^z) = max(z, 0) + log(1 + t), t = e^-|z|, by the series of log((1 + s) / (1 - s)) = 2 (s + s^3 / 3 + ..), s = t / (2 + t) <= 1/3,
// cut where its terms pass below 2e-9 of the sum. As close to 64 bits as the library's log1pf (1.3e-7 at most, 2.5e-8 in the mean square) at a
// third of its instructions, which were half of what the kernel issued.
__device__ __forceinline__ float delta_softplus(float z) {
    const float t = expf(-fabsf(z)), d = 2.0f + t;
    const float r = __builtin_amdgcn_rcpf(d);
    float s = t * r;
    s = fmaf(fmaf(-d, s, t), r, s);
    const float y = s * s;
    float sum = fmaf(y, 1.0f / 15.0f, 1.0f / 13.0f);
    sum = fmaf(y, sum, 1.0f / 11.0f);
    sum = fmaf(y, sum, 1.0f / 9.0f);
    sum = fmaf(y, sum, 1.0f / 7.0f);
    sum = fmaf(y, sum, 0.2f);
    sum = fmaf(y, sum, 1.0f / 3.0f);
    sum = fmaf(y * s, sum, s);
    return fmaf(2.0f, sum, fmaxf(z, 0.0f));
}
// 1 / (1 + e^-x), the quotient as a reciprocal and one step of Newton's method (as exact as the division). Below -88.7 the divisor is
// infinite and the step would be infinity times zero: the result is 0, as the division's.
__device__ __forceinline__ float delta_sigmoid(float x) {
    const float d = 1.0f + expf(-x);
    const float r = __builtin_amdgcn_rcpf(d);
    return r == 0.0f ? r : fmaf(fmaf(-d, r, 1.0f), r, r);
}

// What up to REACH tokens from token j on see of its key: over the channels at .. at + 3, at + stride .., summed over the sixteen lanes of
// `part`. vectors: q | k | g, [16][D] each.
template <int REACH>
__device__ __forceinline__ void delta_meet(const float* vectors, int D, int at, int stride, int j, int part, float (*keys_met)[CHUNK],
                                           float (*reads_met)[CHUNK]) {
    float kk[REACH], qk[REACH];                         // of token j + d
#pragma unroll
    for (int d = 0; d < REACH; ++d) kk[d] = qk[d] = 0.0f;
    for (; at < D; at += stride) {
        f32x4 reach;                                    // k_j times the decays behind token j
#pragma unroll
        for (int d = 0; d < REACH; ++d) {
            if (d % 4 == 0) __builtin_amdgcn_sched_barrier(0);               // (all rows asked for at once take every register)
            const int i = j + d < CHUNK ? j + d : CHUNK - 1;
            const f32x4 qi = *reinterpret_cast<const f32x4*>(vectors + i * D + at);
            const f32x4 ki = *reinterpret_cast<const f32x4*>(vectors + (CHUNK + i) * D + at);
            if (d == 0) {
                reach = ki;
            } else {
                const f32x4 gi = *reinterpret_cast<const f32x4*>(vectors + (2 * CHUNK + i) * D + at);
#pragma unroll
                for (int e = 0; e < 4; ++e) reach[e] *= gi[e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (d > 0) kk[d] = fmaf(ki[e], reach[e], kk[d]);
                qk[d] = fmaf(qi[e], reach[e], qk[d]);
            }
        }
    }
#pragma unroll
    for (int d = 0; d < REACH; ++d) {
        const float keys = delta_row_sum(kk[d]), reads = delta_row_sum(qk[d]);
        if (part == 0 && j + d < CHUNK) {
            keys_met[j + d][j] = keys;
            reads_met[j + d][j] = reads;
        }
    }
}

// A workgroup per (chunk, head), a thread per channel of q, of k, of the decays and of v, which walks the sixteen tokens. FEW: at most four
// taps, a channel's inputs are loaded once. The chunk's sums L and A (q in place of k_i) are formed by 256 or 512 threads, token j and a
// sixteenth (or half of one) of the channels each, from copies in LDS; then the threads of k and v solve a column of the triangular
// system each. Bound by the instructions it issues and by the latency of its phases: one chunk alone takes 13 us, 1,120 workgroups 43 us.
// With q, k and g of a channel on one thread (half the threads) it took 22 and 56 us.
template <bool FEW>
__global__ __launch_bounds__(1024) void delta_chunk_kernel(
    const float* __restrict__ proj, int proj_stride, int beta_col, const float* __restrict__ a, int a_stride, const float* __restrict__ taps,
    const float* __restrict__ conv_state, const float* __restrict__ A_log, const float* __restrict__ dt_bias,
    const int32_t* __restrict__ seg_row0, const int32_t* __restrict__ seg_slot, float* __restrict__ packets, int segments,
    int heads, int kv_heads, int dim, int vdim, int taps_count, int decay_per_head) {
    extern __shared__ __attribute__((aligned(16))) float vectors[];     // q | k | g, [16][D] each
    __shared__ __attribute__((aligned(16))) float keys_met[2][CHUNK][CHUNK], reads_met[2][CHUNK][CHUNK];
    __shared__ float strength[CHUNK], factor[2 * CHUNK];
    const int chunk = blockIdx.x, head = blockIdx.y, tid = threadIdx.x;
    int seg = 0;
    for (int last = segments - 1; seg < last;) {        // the last segment that begins at or before this chunk
        const int mid = (seg + last + 1) >> 1;
        if (seg_row0[mid] / CHUNK + mid <= chunk) seg = mid;
        else last = mid - 1;
    }
    const int first = seg_row0[seg], count = seg_row0[seg + 1] - first;
    const int before_rows = (chunk - first / CHUNK - seg) * CHUNK;
    if (before_rows >= count) return;                   // a place that this segment does not need
    const int tokens = count - before_rows < CHUNK ? count - before_rows : CHUNK;
    const int row0 = first + before_rows;
    const int D = delta_key_width(dim), V = delta_value_width(vdim);
    const int group = heads / kv_heads, channels = 2 * kv_heads * dim + heads * vdim, keep = taps_count - 1;
    const float* memory = conv_state + (size_t)seg_slot[seg] * channels * keep;

    // silu of the convolution of channel c, the chunk's sixteen tokens (zero behind the segment's end)
    auto convolve = [&](int c, float (&y)[CHUNK]) {
        const float* column = proj + c;
        if constexpr (FEW) {
            float x[CHUNK + 3], w[4];                   // x[i]: the input of row row0 - 3 + i
#pragma unroll
            for (int b = 0; b < 4; ++b) w[b] = taps[(size_t)c * taps_count + (b < taps_count ? keep - b : 0)];       // looks b rows back
#pragma unroll
            for (int i = 0; i < CHUNK; ++i) x[i + 3] = column[(size_t)(row0 + (i < tokens ? i : tokens - 1)) * proj_stride];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                x[i] = 0.0f;
                if (before_rows > 0) x[i] = column[(size_t)(row0 - 3 + i) * proj_stride];
                else if (3 - i <= keep) x[i] = memory[(size_t)c * keep + keep - 3 + i];
            }
#pragma unroll
            for (int i = 0; i < CHUNK; ++i) {
                float sum = 0.0f;
#pragma unroll
                for (int b = 3; b >= 0; --b)
                    if (b < taps_count) sum = fmaf(w[b], x[i + 3 - b], sum);
                y[i] = i < tokens ? sum * delta_sigmoid(sum) : 0.0f;
            }
        } else {
#pragma unroll
            for (int i = 0; i < CHUNK; ++i) {
                y[i] = 0.0f;
                if (i >= tokens) continue;
                float sum = 0.0f;
                for (int j = 0; j < taps_count; ++j) {
                    const int at = before_rows + i - (keep - j);
                    const float x = at >= 0 ? column[(size_t)(first + at) * proj_stride] : memory[(size_t)c * keep + keep + at];
                    sum = fmaf(taps[(size_t)c * taps_count + j], x, sum);
                }
                y[i] = sum * delta_sigmoid(sum);
            }
        }
    };

    const int kind = tid / D < 3 ? tid / D : 3;         // q, k, decay, v (whole waves: D is a multiple of 64)
    const int c = tid - kind * D;
    float x[CHUNK];                                     // this channel's values: of k and v they are worked on below
#pragma unroll
    for (int i = 0; i < CHUNK; ++i) x[i] = kind == 2 ? 1.0f : 0.0f;
    if (kind == 2) {
        if (c < dim) {
            const int at = decay_per_head ? head : head * dim + c;
            const float rate = expf(A_log[head]), bias = dt_bias[at];
#pragma unroll
            for (int i = 0; i < CHUNK; ++i) x[i] = a[(size_t)(row0 + (i < tokens ? i : tokens - 1)) * a_stride + at];
#pragma unroll
            for (int i = 0; i < CHUNK; ++i) x[i] = i < tokens ? expf(-rate * delta_softplus(x[i] + bias)) : 1.0f;
        }
    } else if (c < (kind == 3 ? vdim : dim)) {
        convolve(kind == 3 ? 2 * kv_heads * dim + head * vdim + c : (kind * kv_heads + head / group) * dim + c, x);
    }
    if (kind < 3) {
#pragma unroll
        for (int i = 0; i < CHUNK; ++i) vectors[(kind * CHUNK + i) * D + c] = x[i];
    }
    if (tid < CHUNK) strength[tid] = tid < tokens ? delta_sigmoid(proj[(size_t)(row0 + tid) * proj_stride + beta_col + head]) : 0.0f;
    __syncthreads();

    // unit vectors: one factor per token for q and for k
    const int lane = tid & 63;
    for (int p = tid >> 6; p < 2 * CHUNK; p += blockDim.x >> 6) {
        float sum = 0.0f;
        for (int at = lane; at < D; at += 64) sum += vectors[p * D + at] * vectors[p * D + at];
        sum = fw_quad_sum(delta_row_sum(sum));
        if (lane == 0) factor[p] = 1.0f / sqrtf(sum + 1e-6f) * (p < CHUNK ? 1.0f / sqrtf((float)dim) : 1.0f);
    }
    // what the tokens' keys and queries see of the keys before them
    const int halves = blockDim.x >= 512 && D > 64 ? 2 : 1;
    if (tid < 256 * halves) {
        const int half = tid >> 8, j = (tid >> 4) & 15, part = tid & 15;
        float(*keys)[CHUNK] = keys_met[half], (*reads)[CHUNK] = reads_met[half];
        switch (__builtin_amdgcn_readfirstlane((tid >> 6) & 3)) {           // a wave's first token of four decides how many lie behind it
            case 0: delta_meet<16>(vectors, D, part * 4 + half * 64, 64 * halves, j, part, keys, reads); break;
            case 1: delta_meet<12>(vectors, D, part * 4 + half * 64, 64 * halves, j, part, keys, reads); break;
            case 2: delta_meet<8>(vectors, D, part * 4 + half * 64, 64 * halves, j, part, keys, reads); break;
            default: delta_meet<4>(vectors, D, part * 4 + half * 64, 64 * halves, j, part, keys, reads); break;
        }
    }
    __syncthreads();
    for (int item = tid; item < 256; item += blockDim.x) {
        const int i = item >> 4, j = item & 15;
        if (j > i) continue;
        const float keys = halves > 1 ? keys_met[0][i][j] + keys_met[1][i][j] : keys_met[0][i][j];
        const float reads = halves > 1 ? reads_met[0][i][j] + reads_met[1][i][j] : reads_met[0][i][j];
        keys_met[0][i][j] = keys * factor[CHUNK + i] * factor[CHUNK + j];
        reads_met[0][i][j] = reads * factor[i] * factor[CHUNK + j];
    }
    __syncthreads();

    // Every column of the system by forward substitution: key channel c has G_i k_i on its right side and gives W, value
    // channel has v_i and gives Uv. Then what the tokens read.
    if (kind == 0 || kind == 2) return;
    const bool key = kind == 1;
    if (!key && c >= V) return;
    float* packet = packets + ((size_t)chunk * heads + head) * (49 * D + 32 * V);
    float read[CHUNK];
#pragma unroll
    for (int i = 0; i < CHUNK; ++i) read[i] = 0.0f;
    if (key) {
        float reach = 1.0f;
        f32x4 written[CHUNK / 4];
#pragma unroll
        for (int i = 0; i < CHUNK; ++i) x[i] *= factor[CHUNK + i];
#pragma unroll
        for (int i = CHUNK - 1; i >= 0; --i) {
            written[i / 4][i % 4] = x[i] * reach;
            reach *= vectors[(2 * CHUNK + i) * D + c];
        }
#pragma unroll
        for (int i = 0; i < CHUNK / 4; ++i) *reinterpret_cast<f32x4*>(packet + 32 * D + c * CHUNK + 4 * i) = written[i];
        packet[48 * D + c] = reach;
        reach = 1.0f;
#pragma unroll
        for (int i = 0; i < CHUNK; ++i) {
            reach *= vectors[(2 * CHUNK + i) * D + c];
            x[i] *= reach;
            read[i] = vectors[i * D + c] * factor[i] * reach;
        }
    }
#pragma unroll
    for (int i = 0; i < CHUNK; ++i) {
        f32x4 row[CHUNK / 4];
#pragma unroll
        for (int j = 0; j < i; j += 4) row[j / 4] = *reinterpret_cast<const f32x4*>(&keys_met[0][i][j]);
        float rest = 0.0f;
#pragma unroll
        for (int j = 0; j < i; ++j) rest = fmaf(row[j / 4][j % 4], x[j], rest);
        x[i] = strength[i] * (x[i] - rest);
    }
    const float sign = key ? -1.0f : 1.0f;
#pragma unroll
    for (int i = 0; i < CHUNK; ++i) {
        f32x4 row[CHUNK / 4];
#pragma unroll
        for (int j = 0; j <= i; j += 4) row[j / 4] = *reinterpret_cast<const f32x4*>(&reads_met[0][i][j]);
        float seen = 0.0f;
#pragma unroll
        for (int j = 0; j <= i; ++j) seen = fmaf(row[j / 4][j % 4], x[j], seen);
        read[i] = fmaf(sign, seen, read[i]);
    }
    if (key) {
        float* to = packet + (c >> 4) * 256 + (c & 15);
#pragma unroll
        for (int i = 0; i < CHUNK; ++i) {
            to[i * 16] = x[i];
            to[16 * D + i * 16] = read[i];
        }
    } else {
        float* to = packet + 49 * D + c * CHUNK;
#pragma unroll
        for (int i = 0; i < CHUNK; i += 4) {
            *reinterpret_cast<f32x4*>(to + i) = f32x4{x[i], x[i + 1], x[i + 2], x[i + 3]};
            *reinterpret_cast<f32x4*>(to + 16 * V + i) = f32x4{read[i], read[i + 1], read[i + 2], read[i + 3]};
        }
    }
}

// A workgroup per (segment, head, sixteen value channels); wave w holds KT tiles of S, key channels 16 (w KT + t) .. + 15, as a product
// of the matrix instruction leaves it: lane l has column l % 16, rows 4 (l / 16) + r. That is also how the instruction reads its
// second operand (with the k of instruction r being 4 (l / 16) + r), so S goes from product to product without a move, and so does u. The
// operands of a chunk are read by one wave each, straight into registers, AHEAD chunks early. The four waves' parts of W S0 meet in LDS
// (one barrier a chunk); what a chunk's tokens read leaves a chunk later. 0.97 us a chunk at KT 2, of which the 24 matrix instructions of
// a wave are 0.32; without its loads the walk would take 0.7. One chunk more or two more on the way changed nothing.
template <int KT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(KT <= 2 ? 2 : 1, KT <= 2 ? 2 : 1))) void delta_walk_kernel(
    const float* __restrict__ packets, float* __restrict__ state, float* __restrict__ out, const int32_t* __restrict__ seg_row0,
    const int32_t* __restrict__ seg_slot, int heads, int dim, int vdim, int runs_whole) {
    constexpr int D = KT * 64, AHEAD = 3;
    __shared__ __attribute__((aligned(16))) f32x4 seen_parts[2][4][64], read_parts[2][4][64];
    const int seg = blockIdx.x, head = blockIdx.y, block = blockIdx.z;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 15, quad = lane >> 4;
    const int V = delta_value_width(vdim);
    const int first = seg_row0[seg], count = seg_row0[seg + 1] - first;
    const int chunks = (count + CHUNK - 1) / CHUNK;
    if (chunks == 0) return;
    const size_t stride = (size_t)heads * (49 * D + 32 * V);            // from a chunk's packet to the next one's
    const float* packet = packets + ((size_t)(first / CHUNK + seg) * heads + head) * (49 * D + 32 * V);

    struct Operands {
        f32x4 w[KT], q[KT], k[KT], g[KT], uv;
        float ov;
    };
    // this thread's read-out of a chunk: token 4 wave + tid % 4, column tid / 4 % 16
    const int out_token = wave * 4 + (tid & 3), out_col = (tid >> 2) & 15;
    // (places within a packet as 32-bit offsets of the lane beside an address that all lanes share)
    const uint32_t at_tile = wave * KT * 256 + col * 16 + quad * 4, at_decay = 48 * D + wave * KT * 16 + quad * 4;
    const uint32_t at_uv = 49 * D + (block * 16 + col) * CHUNK + quad * 4, at_ov = 49 * D + 16 * V + (block * 16 + out_col) * CHUNK + out_token;
    auto ask = [&](Operands& f, int chunk) {
        const float* from = packet + (size_t)(chunk < chunks ? chunk : chunks - 1) * stride;       // (behind the end: read again, not used)
#pragma unroll
        for (int t = 0; t < KT; ++t) {
            f.w[t] = *reinterpret_cast<const f32x4*>(from + t * 256 + at_tile);
            f.q[t] = *reinterpret_cast<const f32x4*>(from + 16 * D + t * 256 + at_tile);
            f.k[t] = *reinterpret_cast<const f32x4*>(from + 32 * D + t * 256 + at_tile);
            f.g[t] = *reinterpret_cast<const f32x4*>(from + t * 16 + at_decay);
        }
        f.uv = *reinterpret_cast<const f32x4*>(from + at_uv);
        f.ov = from[at_ov];
    };
    Operands held[AHEAD];
#pragma unroll
    for (int n = 0; n < AHEAD; ++n) ask(held[n], n);

    const bool live = block * 16 + col < vdim;
    float* mine = state + (((size_t)seg_slot[seg] * heads + head) * vdim + (live ? block * 16 + col : 0)) * dim;
    f32x4 S[KT];
#pragma unroll
    for (int t = 0; t < KT; ++t) {
        const int c = (wave * KT + t) * 16 + quad * 4;
        S[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if (!live) continue;
        if (runs_whole) {
            if (c < dim) S[t] = *reinterpret_cast<const f32x4*>(mine + c);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (c + e < dim) S[t][e] = mine[c + e];
        }
    }
    float* out_at = out + (size_t)first * heads * vdim + (size_t)head * vdim + block * 16 + out_col;
    const bool out_live = block * 16 + out_col < vdim;
    float ov_before = 0.0f;
    // a chunk's read-outs from its parts in LDS (none ahead of the first)
    const float* parts = reinterpret_cast<const float*>(read_parts) + tid;
    auto leave = [&](int chunk, float sum) {
        const int token = chunk * CHUNK + out_token;
        if (out_live && (unsigned)token < (unsigned)count) out_at[(size_t)token * heads * vdim] = ov_before + sum;
    };
    auto step = [&](Operands& f, int chunk, bool more) {
        const int here = chunk & 1, other = (here ^ 1) * 1024;
        f32x4 seen[2], read[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) seen[t] = read[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int t = 0; t < KT; ++t) seen[t & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.w[t][r], S[t][r], seen[t & 1], 0, 0, 0);
        seen_parts[here][wave][lane] = KT > 1 ? seen[0] + seen[1] : seen[0];
        __builtin_amdgcn_sched_barrier(0);              // what the tokens read waits behind the chain, and covers LDS's latency
        fw_lds_barrier();
        const f32x4 p0 = seen_parts[here][0][lane], p1 = seen_parts[here][1][lane], p2 = seen_parts[here][2][lane], p3 = seen_parts[here][3][lane];
        const float r0 = parts[other], r1 = parts[other + 256], r2 = parts[other + 512], r3 = parts[other + 768];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int t = 0; t < KT; ++t) read[t & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.q[t][r], S[t][r], read[t & 1], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < KT; ++t) S[t] *= f.g[t];
        __builtin_amdgcn_sched_barrier(0);
        const f32x4 u = f.uv - (((p0 + p1) + p2) + p3);
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int t = 0; t < KT; ++t) S[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.k[t][r], u[r], S[t], 0, 0, 0);
        read_parts[here][wave][lane] = KT > 1 ? read[0] + read[1] : read[0];
        leave(chunk - 1, ((r0 + r1) + r2) + r3);
        ov_before = f.ov;
        if (more) ask(f, chunk + AHEAD);
        fw_mfma_drain();
    };
    // (whole turns without a condition: where paths of different length meet, the compiler waits for loads as if the shortest had been taken)
    int chunk = 0;
    for (; chunk + AHEAD <= chunks; chunk += AHEAD)
#pragma unroll
        for (int n = 0; n < AHEAD; ++n) step(held[n], chunk + n, true);
#pragma unroll
    for (int n = 0; n < AHEAD - 1; ++n)
        if (chunk + n < chunks) step(held[n], chunk + n, false);
    fw_lds_barrier();
    const int last = ((chunks - 1) & 1) * 1024;
    leave(chunks - 1, ((parts[last] + parts[last + 256]) + parts[last + 512]) + parts[last + 768]);
    if (!live) return;
#pragma unroll
    for (int t = 0; t < KT; ++t) {
        const int c = (wave * KT + t) * 16 + quad * 4;
        if (runs_whole) {
            if (c < dim) *reinterpret_cast<f32x4*>(mine + c) = S[t];
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (c + e < dim) mine[c + e] = S[t][e];
        }
    }
}

extern "C" int fw_delta_chunks(const float* proj, int proj_stride, int beta_col, const float* a, int a_stride, const float* taps,
                               float* conv_state, const float* A_log, const float* dt_bias, const int32_t* seg_row0,
                               const int32_t* seg_slot, float* packets, float* state, float* out, int rows, int segments, int heads,
                               int kv_heads, int dim, int vdim, int taps_count, int slots, int decay_per_head, void* stream) {
    FW_REQUIRE(rows >= 0 && segments >= 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0,
               "delta_chunks: heads %d must be a positive multiple of kv heads %d", heads, kv_heads);
    FW_REQUIRE(dim > 0 && dim <= 256 && vdim > 0 && vdim <= 256, "delta_chunks: dim %d and vdim %d must lie in 1..256", dim, vdim);
    FW_REQUIRE(taps_count >= 1 && taps_count <= 17, "delta_chunks: %d taps outside 1..17", taps_count);
    FW_REQUIRE(slots > 0, "delta_chunks: no state slots");
    const int channels = 2 * kv_heads * dim + heads * vdim;
    FW_REQUIRE(proj_stride >= channels && beta_col >= 0 && beta_col + heads <= proj_stride,
               "delta_chunks: the projections' rows (%d wide) do not hold %d channels and %d strengths at %d", proj_stride, channels, heads, beta_col);
    FW_REQUIRE(a_stride >= (decay_per_head ? heads : heads * dim), "delta_chunks: the decays' arguments (%d wide) do not hold %d x %d", a_stride, heads, decay_per_head ? 1 : dim);
    FW_REQUIRE(rows <= 1 << 20 && segments <= 65535 && heads <= 65535, "delta_chunks: too many rows, segments or heads");
    FW_REQUIRE((uintptr_t)packets % 16 == 0, "delta_chunks: the packets must lie at a multiple of 16 bytes");
    if (rows == 0 || segments == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const int D = delta_key_width(dim), V = delta_value_width(vdim);
    const dim3 grid(fw_delta_chunk_slots(rows, segments), heads);
    const int threads = (3 * D + V + 63) & ~63, lds = 3 * CHUNK * D * (int)sizeof(float);
    if (taps_count <= 4)
        delta_chunk_kernel<true><<<grid, threads, lds, s>>>(proj, proj_stride, beta_col, a, a_stride, taps, conv_state, A_log, dt_bias, seg_row0,
                                                            seg_slot, packets, segments, heads, kv_heads, dim, vdim, taps_count, decay_per_head);
    else
        delta_chunk_kernel<false><<<grid, threads, lds, s>>>(proj, proj_stride, beta_col, a, a_stride, taps, conv_state, A_log, dt_bias, seg_row0,
                                                             seg_slot, packets, segments, heads, kv_heads, dim, vdim, taps_count, decay_per_head);
    if (taps_count > 1) fw_launch_conv_state(proj, FW_F32, proj_stride, conv_state, seg_row0, seg_slot, channels, taps_count, segments, s);
    const int runs_whole = dim % 4 == 0 && (uintptr_t)state % 16 == 0;
    const dim3 walk(segments, heads, V / 16);
#define FW_WALK(KT) delta_walk_kernel<KT><<<walk, 256, 0, s>>>(packets, state, out, seg_row0, seg_slot, heads, dim, vdim, runs_whole)
    switch (D / 64) {
        case 1: FW_WALK(1); break;
        case 2: FW_WALK(2); break;
        case 3: FW_WALK(3); break;
        default: FW_WALK(4); break;
    }
#undef FW_WALK
    FW_LAUNCH_CHECK("delta_chunks");
    return 0;
}
