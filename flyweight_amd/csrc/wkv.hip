// A linear recurrence over a matrix state per head with a decay per key channel that the token itself
// forms and a bonus for the current token ("wkv"), and the mixing of a token's input with the input of the
// token before it that stands in front of it. All arithmetic float32, whatever the run's dtype.
//
//   o_t = (S + diag(u) k_t v_t^T)^T r_t = S^T r_t + (sum_c r_t[c] u[c] k_t[c]) v_t
//   S  <- diag(w_t) S + k_t v_t^T,            w_t = exp(-exp(a_t + w0))
//
// S [key channel][value channel] per head and request, zero at a request's start.
#include "fw_common.h"
#include "fw_kernels.h"

// ---- token shift --------------------------------------------------------------------------------
// A workgroup per row. h = x * rsqrt(mean(x^2) + eps) * (w or 1 + w) (norm_weight null: h = x). The row
// before comes from the same step (normed again here: a row is read twice, nothing is kept between
// workgroups) or, for a segment's first row, from the request's slot. out[s][row] = h + (before - h) *
// mu[s]. The workgroup of a segment's FIRST row also moves the slot on to the h of the segment's LAST
// row: it alone reads and writes the slot, each thread its own channels, the read first. A step of few rows
// has several workgroups a row (blockIdx.y), each with channels of its own (and the row's sums of squares once
// more): a single token's mixes are then a few loads deep, not one round of loads after the other.
template <typename T>
__global__ __launch_bounds__(256) void token_shift_mix_kernel(
    const float* __restrict__ x, const float* __restrict__ norm_weight, float eps, int one_centered,
    const float* __restrict__ mu, int mixes, float* __restrict__ last, const int32_t* __restrict__ row_seg,
    const int32_t* __restrict__ seg_row0, const int32_t* __restrict__ seg_slot, T* __restrict__ out, int rows, int hidden) {
    __shared__ float scratch[16];
    const int row = blockIdx.x;
    const int seg = row_seg[row];
    const int first_row = seg_row0[seg], last_row = seg_row0[seg + 1] - 1;
    const bool is_first = row == first_row;
    float* slot = last + (size_t)seg_slot[seg] * hidden;
    auto inverse_rms = [&](const float* source) {
        if (!norm_weight) return 1.0f;
        float sum = 0.0f;
        for (int i = threadIdx.x; i < hidden; i += 256) sum += source[i] * source[i];
        sum = block_sum(sum, scratch);
        return rsqrtf(sum / (float)hidden + eps);
    };
    const float* mine = x + (size_t)row * hidden;
    const float* other = x + (size_t)(is_first ? last_row : row - 1) * hidden;     // a first row: the row that the slot will hold
    const float inv = inverse_rms(mine);
    const float inv_other = (is_first && last_row == row) ? inv : inverse_rms(other);
    for (int i = blockIdx.y * 256 + threadIdx.x; i < hidden; i += 256 * gridDim.y) {
        const float w = norm_weight ? (one_centered ? 1.0f + norm_weight[i] : norm_weight[i]) : 1.0f;
        const float h = mine[i] * inv * w;
        const float h_other = other[i] * inv_other * w;
        float before = h_other;
        if (is_first) {
            before = slot[i];
            slot[i] = h_other;
        }
        for (int s = 0; s < mixes; ++s)
            store_from_float(out, ((size_t)s * rows + row) * hidden + i, fmaf(before - h, mu[(size_t)s * hidden + i], h));
    }
}

// The same for a prompt's rows that lie at 16 bytes: R neighbouring rows to a workgroup. A row to a workgroup read every row and summed its squares
// twice, and brought all of mu (40 KB of five mixes of 2,048 channels) along for it. The sums first, in the order of the kernel above (the same bits), then
// four channels to a thread. Bound by the mixes that it stores. 2,048 rows of 2,048, five mixes 36.6 -> 26.3 us (59 MB).
template <typename T, int R>
__global__ __launch_bounds__(256) void token_shift_mix_rows_kernel(
    const float* __restrict__ x, const float* __restrict__ norm_weight, float eps, int one_centered,
    const float* __restrict__ mu, int mixes, float* __restrict__ last, const int32_t* __restrict__ row_seg,
    const int32_t* __restrict__ seg_row0, const int32_t* __restrict__ seg_slot, T* __restrict__ out, int rows, int hidden) {
    typedef __attribute__((ext_vector_type(4))) float f32x4;
    __shared__ float scratch[2 * R][4];
    const int r0 = blockIdx.x * R, tid = threadIdx.x;
    int row_of[R], other_of[R];
    bool is_first[R];
    float* slot[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        row_of[r] = r0 + r < rows ? r0 + r : rows - 1;
        const int seg = row_seg[row_of[r]];
        is_first[r] = row_of[r] == seg_row0[seg];
        other_of[r] = is_first[r] ? seg_row0[seg + 1] - 1 : row_of[r] - 1;      // a first row: the row that the slot will hold
        slot[r] = last + (size_t)seg_slot[seg] * hidden;
    }
    float inv[R], inv_other[R];
#pragma unroll
    for (int r = 0; r < R; ++r) inv[r] = inv_other[r] = 1.0f;
    if (norm_weight) {
        // a row's neighbour is mostly the row before it here
        auto own = [&](int r) { return !(r > 0 && other_of[r] == row_of[r] - 1) && other_of[r] != row_of[r]; };
        float sum[2 * R] = {};
        for (int i = tid; i < hidden; i += 256)
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const float mine = x[(size_t)row_of[r] * hidden + i];
                sum[r] += mine * mine;
                if (own(r)) {
                    const float other = x[(size_t)other_of[r] * hidden + i];
                    sum[R + r] += other * other;
                }
            }
#pragma unroll
        for (int r = 0; r < 2 * R; ++r) {
            if (r >= R && !own(r - R)) continue;
            const float all = wave_sum(sum[r]);
            if ((tid & 63) == 0) scratch[r][tid >> 6] = all;
        }
        __syncthreads();
        auto inverse = [&](int r) { return rsqrtf((((scratch[r][0] + scratch[r][1]) + scratch[r][2]) + scratch[r][3]) / (float)hidden + eps); };
#pragma unroll
        for (int r = 0; r < R; ++r) {
            inv[r] = inverse(r);
            inv_other[r] = own(r) ? inverse(R + r) : other_of[r] == row_of[r] ? inv[r] : inv[r > 0 ? r - 1 : 0];
        }
    }
    for (int i = tid * 4; i < hidden; i += 1024) {
        f32x4 w = {1.0f, 1.0f, 1.0f, 1.0f};
        if (norm_weight) {
            w = *reinterpret_cast<const f32x4*>(norm_weight + i);
            if (one_centered) w = w + 1.0f;
        }
        f32x4 h[R], apart[R];                                               // apart: what the row before it is more
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (r0 + r >= rows) break;
            const f32x4 mine = *reinterpret_cast<const f32x4*>(x + (size_t)row_of[r] * hidden + i);
            const f32x4 other = *reinterpret_cast<const f32x4*>(x + (size_t)other_of[r] * hidden + i);
            f32x4 before;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                h[r][e] = mine[e] * inv[r] * w[e];
                before[e] = other[e] * inv_other[r] * w[e];
            }
            if (is_first[r]) {
                const f32x4 held = *reinterpret_cast<const f32x4*>(slot[r] + i);
                *reinterpret_cast<f32x4*>(slot[r] + i) = before;
                before = held;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) apart[r][e] = before[e] - h[r][e];
        }
        for (int s = 0; s < mixes; ++s) {
            const f32x4 m = *reinterpret_cast<const f32x4*>(mu + (size_t)s * hidden + i);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (r0 + r >= rows) break;
                f32x4 y;
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] = fmaf(apart[r][e], m[e], h[r][e]);
                T* to = out + ((size_t)s * rows + row_of[r]) * hidden + i;
                if constexpr (sizeof(T) == 4) {
                    *reinterpret_cast<f32x4*>(to) = y;
                } else {
                    *reinterpret_cast<uint2*>(to) = make_uint2((uint32_t)float_to_bf16_bits(y[0]) | ((uint32_t)float_to_bf16_bits(y[1]) << 16),
                                                               (uint32_t)float_to_bf16_bits(y[2]) | ((uint32_t)float_to_bf16_bits(y[3]) << 16));
                }
            }
        }
    }
}

extern "C" int fw_token_shift_mix(const float* x, const float* norm_weight, float eps, int one_centered, const float* mu, int mixes,
                                  float* last, int slots, const int32_t* row_seg, const int32_t* seg_row0, const int32_t* seg_slot,
                                  void* out, int out_dtype, int rows, int segments, int hidden, void* stream) {
    FW_REQUIRE(rows >= 0 && segments >= 0 && hidden > 0 && mixes > 0 && slots > 0, "token_shift_mix: bad sizes rows=%d segments=%d hidden=%d mixes=%d",
               rows, segments, hidden, mixes);
    FW_REQUIRE(rows <= 1 << 20, "token_shift_mix: too many rows (%d)", rows);
    if (rows == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    // beyond 128 rows (up to there several workgroups share a row); four rows to a workgroup while that leaves every compute unit one
    auto lies = [](const void* p) { return (uintptr_t)p % 16 == 0; };
    if (rows > 128 && hidden % 4 == 0 && lies(x) && lies(norm_weight) && lies(mu) && lies(last) && lies(out) && (out_dtype == FW_F32 || out_dtype == FW_BF16)) {
#define FW_ROWS_LAUNCH(T, R) \
    token_shift_mix_rows_kernel<T, R><<<fw_ceil_div(rows, R), 256, 0, s>>>(x, norm_weight, eps, one_centered, mu, mixes, last, row_seg, seg_row0, seg_slot, (T*)out, rows, hidden)
        if (out_dtype == FW_F32) {
            if (rows >= 1024) FW_ROWS_LAUNCH(float, 4);
            else FW_ROWS_LAUNCH(float, 2);
        } else {
            if (rows >= 1024) FW_ROWS_LAUNCH(bf16_t, 4);
            else FW_ROWS_LAUNCH(bf16_t, 2);
        }
#undef FW_ROWS_LAUNCH
        FW_LAUNCH_CHECK("token_shift_mix");
        return 0;
    }
    const int parts = rows <= 128 ? (fw_ceil_div(hidden, 256) < 16 ? fw_ceil_div(hidden, 256) : 16) : 1;
    const dim3 grid(rows, parts);
    if (out_dtype == FW_F32)
        token_shift_mix_kernel<float><<<grid, 256, 0, s>>>(x, norm_weight, eps, one_centered, mu, mixes, last, row_seg, seg_row0, seg_slot,
                                                           (float*)out, rows, hidden);
    else if (out_dtype == FW_BF16)
        token_shift_mix_kernel<bf16_t><<<grid, 256, 0, s>>>(x, norm_weight, eps, one_centered, mu, mixes, last, row_seg, seg_row0, seg_slot,
                                                            (bf16_t*)out, rows, hidden);
    else
        FW_REQUIRE(false, "token_shift_mix: unknown dtype %d", out_dtype);
    FW_LAUNCH_CHECK("token_shift_mix");
    return 0;
}

// out = tanh(x), float32 in, any dtype out
template <typename T>
__global__ void tanh_rows_kernel(const float* __restrict__ x, T* __restrict__ out, long long count) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (long long)gridDim.x * blockDim.x)
        store_from_float(out, (size_t)i, tanhf(x[i]));
}

extern "C" int fw_tanh_rows(const float* x, void* out, int out_dtype, long long count, void* stream) {
    FW_REQUIRE(count >= 0, "tanh_rows: negative count");
    if (count == 0) return 0;
    const int blocks = (int)((count + 255) / 256 > 4096 ? 4096 : (count + 255) / 256);
    if (out_dtype == FW_F32) tanh_rows_kernel<float><<<blocks, 256, 0, (hipStream_t)stream>>>(x, (float*)out, count);
    else if (out_dtype == FW_BF16) tanh_rows_kernel<bf16_t><<<blocks, 256, 0, (hipStream_t)stream>>>(x, (bf16_t*)out, count);
    else FW_REQUIRE(false, "tanh_rows: unknown dtype %d", out_dtype);
    FW_LAUNCH_CHECK("tanh_rows");
    return 0;
}

// ---- the recurrence ------------------------------------------------------------------------------
// Workgroup (segment, head, block of 16 value channels); thread = 16 * column + part: a column of S is
// shared out over the 16 lanes of a row of the wave, RPT neighbouring key channels each (a lane reads its
// channels of r, of k and of the decay from LDS in one access each; channels from dim on hold zeros), so that a head is spread over many compute units: the walk along the tokens is one dependent
// chain per column (a single multiply-add per key channel and token), and only its width can be bought.
// Tokens come in chunks of WKV_CHUNK (32, fewer for wide heads, whose tokens are larger). A chunk's r, k, a
// and its block's 16 values travel from global
// memory into registers while the chunk before is walked; on their way into LDS the decay's two
// exponentials are taken, once per chunk and key channel. A column's sums over key channels (the read-out
// S^T r and the bonus r . (u k), which every column forms for itself) are each thread's own sum and then
// the sixteen lanes', inside the vector unit. The state is read at the segment's start and written at its
// end. Columns of S never meet and the lanes' sums have one fixed order, so the result depends neither on
// how the work is cut nor, tokens being walked in order whatever the segments, on the cut of the sequence.
#define WKV_LANES 16
#define WKV_COLUMNS (256 / WKV_LANES)
template <int CTRL>
__device__ __forceinline__ float wkv_dpp(float x) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float wkv_row_sum(float x) {
    x += wkv_dpp<0xB1>(x);          // quad_perm [1, 0, 3, 2]
    x += wkv_dpp<0x4E>(x);          // quad_perm [2, 3, 0, 1]
    x += wkv_dpp<0x141>(x);         // row_half_mirror
    x += wkv_dpp<0x140>(x);         // row_mirror
    return x;
}

//
// CUT: a workgroup walks a chunk of WKV_ROWS rows of a long segment (chunk_seg, chunk_row0) from a zero state; the state
// behind it goes to local[chunk][head] and the product of its decays per key channel to shrink[chunk][head]. Otherwise a
// workgroup walks a segment, and leaves those of more than long_rows rows alone (long_rows > 0).
#define WKV_ROWS 64
template <int RPT, int WKV_CHUNK, bool CUT>
__global__ __launch_bounds__(256) void wkv_recurrence_kernel(
    const float* __restrict__ r, const float* __restrict__ k, const float* __restrict__ v, int rkv_stride,
    const float* __restrict__ a, int a_stride, const float* __restrict__ w0, const float* __restrict__ u, float* __restrict__ state,
    float* __restrict__ out, const int32_t* __restrict__ seg_row0, const int32_t* __restrict__ seg_slot, int heads, int dim, int long_rows,
    const int32_t* __restrict__ chunk_seg, const int32_t* __restrict__ chunk_row0, float* __restrict__ local, float* __restrict__ shrink) {
    constexpr int DP = WKV_LANES * RPT;                 // key channels as the lanes hold them
    constexpr int TOKEN = 3 * DP + WKV_COLUMNS;         // a staged token: r, k, decay, the block's values
    constexpr int PIECES = (WKV_CHUNK * DP + 255) / 256;    // elements of a chunk's r (and k, and a) per thread, at most
    __shared__ __attribute__((aligned(16))) float staged[WKV_CHUNK * TOKEN];
    __shared__ float results[WKV_CHUNK * WKV_COLUMNS];
    constexpr int VALUE_PIECES = (WKV_CHUNK * WKV_COLUMNS + 255) / 256;     // of the block's values of a chunk per thread
    const int seg = CUT ? chunk_seg[blockIdx.x] : blockIdx.x, head = blockIdx.y, block = blockIdx.z;
    const int own = threadIdx.x / WKV_LANES, part = threadIdx.x % WKV_LANES;
    const int column = block * WKV_COLUMNS + own;
    const bool live = column < dim;
    const int first = CUT ? chunk_row0[blockIdx.x] : seg_row0[seg];
    const int rows = seg_row0[seg + 1] - first, count = CUT && rows > WKV_ROWS ? WKV_ROWS : rows;
    if (!CUT && long_rows > 0 && count > long_rows) return;     // its chunks are walked side by side
    const size_t head_at = (size_t)head * dim;
    // This thread's elements of every chunk: element e = thread + 256 i of the chunk's [tokens][dim] block of r,
    // of k and of a alike (token e / dim, channel e % dim), and one of the block's values (token thread / 16,
    // column thread % 16). A token of -1: no such element.
    int piece_token[PIECES], piece_channel[PIECES];
    float piece_w0[PIECES];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        const int e = threadIdx.x + 256 * i;
        const bool there = e < WKV_CHUNK * dim;
        piece_token[i] = there ? e / dim : -1;
        piece_channel[i] = there ? e % dim : 0;
        piece_w0[i] = w0[head_at + piece_channel[i]];
    }
    const int value_column = block * WKV_COLUMNS + threadIdx.x % WKV_COLUMNS;
    int value_token[VALUE_PIECES];
#pragma unroll
    for (int j = 0; j < VALUE_PIECES; ++j) {
        const int token = (threadIdx.x + 256 * j) / WKV_COLUMNS;
        value_token[j] = (token < WKV_CHUNK && value_column < dim) ? token : -1;
    }
    const int staged_tokens = count < WKV_CHUNK ? count : WKV_CHUNK;        // a decode step stages one token
    for (int i = threadIdx.x; i < staged_tokens * TOKEN; i += 256) staged[i] = 0.0f;
    float held_r[PIECES], held_k[PIECES], held_a[PIECES], held_v[VALUE_PIECES];
    // Loads are unconditional and their addresses plain arithmetic (an element past the chunk's end, or one that
    // this thread does not have, is read from a valid place again and never used): behind a branch the compiler
    // would wait for each load at once, and the next chunk would not travel while this one is walked.
    auto ask = [&](int base) {
        const int last = (count - base < WKV_CHUNK ? count - base : WKV_CHUNK) - 1;
        const float* r0 = r + (size_t)(first + base) * rkv_stride + head_at;
        const float* k0 = k + (size_t)(first + base) * rkv_stride + head_at;
        const float* v0 = v + (size_t)(first + base) * rkv_stride + head_at;
        const float* a0 = a + (size_t)(first + base) * a_stride + head_at;
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            int token = piece_token[i] < 0 ? 0 : piece_token[i];
            token = token < last ? token : last;
            held_r[i] = r0[token * rkv_stride + piece_channel[i]];
            held_k[i] = k0[token * rkv_stride + piece_channel[i]];
            held_a[i] = a0[token * a_stride + piece_channel[i]];
        }
#pragma unroll
        for (int j = 0; j < VALUE_PIECES; ++j) {
            int token = value_token[j] < 0 ? 0 : value_token[j];
            token = token < last ? token : last;
            held_v[j] = v0[token * rkv_stride + (value_token[j] < 0 ? 0 : value_column)];
        }
    };
    auto put = [&](int base) {
        const int tokens = count - base < WKV_CHUNK ? count - base : WKV_CHUNK;
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const float decay = expf(-expf(held_a[i] + piece_w0[i]));
            if (piece_token[i] >= 0 && piece_token[i] < tokens) {
                float* to = staged + piece_token[i] * TOKEN + piece_channel[i];
                to[0] = held_r[i];
                to[DP] = held_k[i];
                to[2 * DP] = decay;
            }
        }
#pragma unroll
        for (int j = 0; j < VALUE_PIECES; ++j)
            if (value_token[j] >= 0 && value_token[j] < tokens) staged[value_token[j] * TOKEN + 3 * DP + threadIdx.x % WKV_COLUMNS] = held_v[j];
    };
    ask(0);
    float* mine = (CUT ? local + ((size_t)blockIdx.x * heads + head) * dim * dim
                       : state + ((size_t)seg_slot[seg] * heads + head) * dim * dim) + (live ? column : 0);
    float product = 1.0f;       // CUT, the first block: of this thread's channel's decays
    float S[RPT], bonus[RPT];
#pragma unroll
    for (int t = 0; t < RPT; ++t) {
        const int key = part * RPT + t;
        S[t] = (!CUT && live && key < dim) ? mine[(size_t)key * dim] : 0.0f;
        bonus[t] = key < dim ? u[head_at + key] : 0.0f;
    }
    __syncthreads();        // the zeros are in place
    put(0);
    __syncthreads();
    // The state and the bonus have arrived here, for the compiler too: their first use being inside the loop, every token waited
    // for all loads in flight, the next chunk's among them. (Not with sixteen channels a lane: 1,024 rows 719 us so, 683 without.)
    if constexpr (RPT < 16) {
#pragma unroll
        for (int t = 0; t < RPT; ++t) asm volatile("" : "+v"(S[t]), "+v"(bonus[t]));
    }
    for (int base = 0; base < count; base += WKV_CHUNK) {
        const int tokens = count - base < WKV_CHUNK ? count - base : WKV_CHUNK;
        const bool more = base + WKV_CHUNK < count;
        if (more) ask(base + WKV_CHUNK);
        // a token's operands are read from LDS while the token before it is worked on
        float r_next[RPT], k_next[RPT], w_next[RPT], v_next;
        auto fetch = [&](int token) {
            const float* t0 = staged + token * TOKEN;
#pragma unroll
            for (int t = 0; t < RPT; ++t) {
                r_next[t] = t0[part * RPT + t];
                k_next[t] = t0[DP + part * RPT + t];
                w_next[t] = t0[2 * DP + part * RPT + t];
            }
            v_next = t0[3 * DP + own];
        };
        fetch(0);
        for (int token = 0; token < tokens; ++token) {
            const float value = v_next;
            float read = 0.0f, ruk = 0.0f;
#pragma unroll
            for (int t = 0; t < RPT; ++t) {
                read = fmaf(r_next[t], S[t], read);
                ruk = fmaf(r_next[t] * bonus[t], k_next[t], ruk);
                S[t] = fmaf(w_next[t], S[t], k_next[t] * value);
            }
            fetch(token + 1 < staged_tokens ? token + 1 : token);       // (behind the chunk's last token: read again, not used)
            read = wkv_row_sum(read);
            ruk = wkv_row_sum(ruk);
            if (part == 0) results[token * WKV_COLUMNS + own] = fmaf(ruk, value, read);
        }
        // (barriers that order LDS traffic only: the next chunk's loads stay in flight across them)
        fw_lds_barrier();
        // the chunk's read-outs leave together: a token's 16 columns side by side
        for (int i = threadIdx.x; i < tokens * WKV_COLUMNS; i += 256) {
            const int token = i / WKV_COLUMNS, c = i % WKV_COLUMNS;
            if (block * WKV_COLUMNS + c < dim)
                out[((size_t)first + base + token) * heads * dim + head_at + block * WKV_COLUMNS + c] = results[i];
        }
        if (CUT && block == 0 && threadIdx.x < dim)
            for (int token = 0; token < tokens; ++token) product *= staged[token * TOKEN + 2 * DP + threadIdx.x];
        if constexpr (CUT) fw_lds_barrier();
        if (more) put(base + WKV_CHUNK);
        fw_lds_barrier();
    }
    if (CUT && block == 0 && threadIdx.x < dim) shrink[((size_t)blockIdx.x * heads + head) * dim + threadIdx.x] = product;
    if (live) {
#pragma unroll
        for (int t = 0; t < RPT; ++t) {
            const int key = part * RPT + t;
            if (key < dim) mine[(size_t)key * dim] = S[t];
        }
    }
}

// ---- a long segment in chunks ---------------------------------------------------------------------
// A segment's serial walk is 0.2 us a row on heads x dim / 16 workgroups, whatever the chip could do beside it. Cut into chunks
// of WKV_ROWS rows, the walks run side by side from zero states (the kernel above, CUT); with P_t the product of the
// chunk's decays before row t and S_in the state ahead of the chunk,
//     o_t += S_in^T (P_t r_t);      S_out = diag(shrink) S_in + local
// Bound by the walks' instructions once the chip is full of them. 2,048 rows of 32 heads of 64 channels: 401 us in order ->
// 111 us (the walks) + 14 (the states) + 21 (the read-outs, which read and write every output once more).

// local[chunk] becomes the state ahead of the chunk, the slot moves on to the state behind the segment. A thread per element of
// (segment, head): loads and one multiply-add per chunk, eight chunks asked for at once.
__global__ __launch_bounds__(256) void wkv_chunk_state_kernel(float* __restrict__ local, const float* __restrict__ shrink, float* __restrict__ state,
                                                              const int32_t* __restrict__ seg_chunk0, const int32_t* __restrict__ seg_slot,
                                                              int heads, int dim) {
    const int seg = blockIdx.x, head = blockIdx.y;
    const int begin = seg_chunk0[seg], chunks = seg_chunk0[seg + 1] - begin;
    const int i = blockIdx.z * 256 + threadIdx.x;
    if (chunks <= 0 || i >= dim * dim) return;
    float* slot = state + ((size_t)seg_slot[seg] * heads + head) * dim * dim + i;
    float* at = local + ((size_t)begin * heads + head) * dim * dim + i;
    const float* decay = shrink + ((size_t)begin * heads + head) * dim + i / dim;
    const size_t step = (size_t)heads * dim * dim, decay_step = (size_t)heads * dim;
    float S = *slot;
    for (int c = 0; c < chunks; c += 8) {
        float own[8], by[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int chunk = c + u < chunks ? c + u : chunks - 1;
            own[u] = at[(size_t)chunk * step];
            by[u] = decay[(size_t)chunk * decay_step];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (c + u >= chunks) break;
            at[(size_t)(c + u) * step] = S;
            S = fmaf(by[u], S, own[u]);
        }
    }
    *slot = S;
}

// out[t] += S_in^T (P_t r_t) of a chunk and head. The threads form P_t r_t in LDS, DP channels by 256 / DP runs of rows: a run's
// decays first (their product tells the later runs where to start), then its rows. The product runs on the matrix cores in
// float32 (v_mfma_f32_32x32x2f32), a 32 x 32 tile a wave at a time; a step takes eight channels, lanes 0..31 the first four,
// lanes 32..63 the next four. S_in comes straight from memory.
typedef __attribute__((ext_vector_type(16))) float wkv_f32x16;
typedef __attribute__((ext_vector_type(4))) float wkv_f32x4;
template <int DP>
__global__ __launch_bounds__(256) void wkv_chunk_read_kernel(const float* __restrict__ r, int rkv_stride, const float* __restrict__ a, int a_stride,
                                                             const float* __restrict__ w0, const float* __restrict__ local, float* __restrict__ out,
                                                             const int32_t* __restrict__ chunk_seg, const int32_t* __restrict__ chunk_row0,
                                                             const int32_t* __restrict__ seg_row0, int heads, int dim) {
    constexpr int RUNS = 256 / DP, RUN = WKV_ROWS / RUNS, PITCH = DP + 4;
    extern __shared__ __attribute__((aligned(16))) float scaled[];      // [WKV_ROWS][PITCH], then the runs' products [RUNS][DP]
    float* products = scaled + WKV_ROWS * PITCH;
    const int chunk = blockIdx.x, head = blockIdx.y;
    const int row0 = chunk_row0[chunk], end = seg_row0[chunk_seg[chunk] + 1];
    const int tokens = end - row0 < WKV_ROWS ? end - row0 : WKV_ROWS;
    const size_t head_at = (size_t)head * dim;
    const int channel = threadIdx.x % DP, run = threadIdx.x / DP;
    const int safe = channel < dim ? channel : dim - 1;
    float decay[RUN], query[RUN];
#pragma unroll
    for (int t = 0; t < RUN; ++t) {                     // rows past the end: the last one again, not stored
        const int token = run * RUN + t < tokens ? run * RUN + t : tokens - 1;
        decay[t] = a[(size_t)(row0 + token) * a_stride + head_at + safe];
        query[t] = r[(size_t)(row0 + token) * rkv_stride + head_at + safe];
    }
    const float base = w0[head_at + safe];
    float product = 1.0f;
#pragma unroll
    for (int t = 0; t < RUN; ++t) {
        decay[t] = expf(-expf(decay[t] + base));
        product *= decay[t];
    }
    products[run * DP + channel] = product;
    __syncthreads();
    float before = 1.0f;
    for (int u = 0; u < run; ++u) before *= products[u * DP + channel];
#pragma unroll
    for (int t = 0; t < RUN; ++t) {
        scaled[(run * RUN + t) * PITCH + channel] = channel < dim ? query[t] * before : 0.0f;
        before *= decay[t];
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, half = lane >> 5, within = lane & 31;
    const float* S_in = local + ((size_t)chunk * heads + head) * dim * dim;
    const int tiles = WKV_ROWS / 32 * ((dim + 31) / 32);
    for (int tile = wave; tile < tiles; tile += 4) {
        const int token0 = tile % (WKV_ROWS / 32) * 32, col = tile / (WKV_ROWS / 32) * 32 + within;
        const int from = col < dim ? col : dim - 1;
        float* to = out + (size_t)(row0 + token0) * heads * dim + head_at + col;
        const size_t step = (size_t)heads * dim;
        float old[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int t = 8 * (i >> 2) + 4 * half + (i & 3);
            old[i] = token0 + t < tokens && col < dim ? to[(size_t)t * step] : 0.0f;
        }
        wkv_f32x16 acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
        const float* rows = scaled + (token0 + within) * PITCH + 4 * half;
#pragma unroll
        for (int c = 0; c < DP; c += 8) {
            const wkv_f32x4 x = *reinterpret_cast<const wkv_f32x4*>(rows + c);
            float b[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int key = c + 4 * half + e;       // (channels past dim meet zeros; they are read at the last one)
                b[e] = S_in[(size_t)(key < dim ? key : dim - 1) * dim + from];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e], b[e], acc, 0, 0, 0);
        }
        fw_mfma_drain();
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int t = 8 * (i >> 2) + 4 * half + (i & 3);
            if (token0 + t < tokens && col < dim) to[(size_t)t * step] = old[i] + acc[i];
        }
    }
}

extern "C" int fw_wkv_chunk_plan(void) { return WKV_ROWS; }

extern "C" int fw_wkv_recurrence(const float* r, const float* k, const float* v, int rkv_stride, const float* a, int a_stride,
                                 const float* w0, const float* u, float* state, int slots, float* out, const int32_t* seg_row0,
                                 const int32_t* seg_slot, int rows, int segments, int heads, int dim, const int32_t* chunk_seg,
                                 const int32_t* chunk_row0, const int32_t* seg_chunk0, int chunks, int long_rows, int all_long,
                                 float* workspace, void* stream) {
    FW_REQUIRE(rows >= 0 && segments >= 0 && heads > 0 && heads <= 65535 && slots > 0, "wkv_recurrence: bad sizes rows=%d segments=%d heads=%d", rows, segments, heads);
    FW_REQUIRE(dim >= 1 && dim <= 256, "wkv_recurrence: a head of %d channels (1..256)", dim);
    FW_REQUIRE(rkv_stride >= heads * dim && a_stride >= heads * dim, "wkv_recurrence: rows of %d / %d values do not hold %d heads of %d", rkv_stride, a_stride, heads, dim);
    FW_REQUIRE(chunks >= 0 && (chunks == 0 || (chunk_seg && chunk_row0 && seg_chunk0 && workspace && long_rows > 0)),
               "wkv_recurrence: chunks come with their places, a workspace and the length from which they are used");
    if (rows == 0 || segments == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    float* shrink = workspace ? workspace + (size_t)chunks * heads * dim * dim : nullptr;
#define FW_WKV_LAUNCH(RPT, CHUNK, CUT)                                                                                                     \
    wkv_recurrence_kernel<RPT, CHUNK, CUT><<<dim3(CUT ? chunks : segments, heads, (dim + WKV_COLUMNS - 1) / WKV_COLUMNS), 256, 0, s>>>(    \
        r, k, v, rkv_stride, a, a_stride, w0, u, state, out, seg_row0, seg_slot, heads, dim, chunks > 0 ? long_rows : 0, chunk_seg,        \
        chunk_row0, workspace, shrink)
    if (chunks == 0 || !all_long) {
        // (the chunk's length changes what is staged together, not one sum: steps of single tokens take short chunks,
        // whose bookkeeping at the start is a few loads)
        const bool few = rows <= 4 * segments;
        if (dim <= 16) { if (few) FW_WKV_LAUNCH(1, 4, false); else FW_WKV_LAUNCH(1, 32, false); }
        else if (dim <= 32) { if (few) FW_WKV_LAUNCH(2, 4, false); else FW_WKV_LAUNCH(2, 32, false); }
        else if (dim <= 64) { if (few) FW_WKV_LAUNCH(4, 4, false); else FW_WKV_LAUNCH(4, 32, false); }
        else if (dim <= 128) FW_WKV_LAUNCH(8, 8, false);
        else FW_WKV_LAUNCH(16, 4, false);
        FW_LAUNCH_CHECK("wkv_recurrence");
    }
    if (chunks == 0) return 0;
    if (dim <= 16) FW_WKV_LAUNCH(1, 32, true);
    else if (dim <= 32) FW_WKV_LAUNCH(2, 32, true);
    else if (dim <= 64) FW_WKV_LAUNCH(4, 32, true);
    else if (dim <= 128) FW_WKV_LAUNCH(8, 8, true);
    else FW_WKV_LAUNCH(16, 4, true);
#undef FW_WKV_LAUNCH
    FW_LAUNCH_CHECK("wkv_recurrence (chunks)");
    wkv_chunk_state_kernel<<<dim3(segments, heads, fw_ceil_div(dim * dim, 256)), 256, 0, s>>>(workspace, shrink, state, seg_chunk0, seg_slot, heads, dim);
    FW_LAUNCH_CHECK("wkv_recurrence (states)");
#define FW_WKV_READ(DP)                                                                                                                 \
    wkv_chunk_read_kernel<DP><<<dim3(chunks, heads), 256, (WKV_ROWS * (DP + 4) + 256) * sizeof(float), s>>>(r, rkv_stride, a, a_stride, \
        w0, workspace, out, chunk_seg, chunk_row0, seg_row0, heads, dim)
    if (dim <= 64) FW_WKV_READ(64);
    else if (dim <= 128) FW_WKV_READ(128);
    else {
        static bool configured = false;
        if (!configured) {
            hipError_t status = hipFuncSetAttribute((const void*)wkv_chunk_read_kernel<256>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                    (WKV_ROWS * 260 + 256) * sizeof(float));
            FW_REQUIRE(status == hipSuccess, "wkv_recurrence: cannot reserve LDS: %s", hipGetErrorString(status));
            configured = true;
        }
        FW_WKV_READ(256);
    }
#undef FW_WKV_READ
    FW_LAUNCH_CHECK("wkv_recurrence (read)");
    return 0;
}
