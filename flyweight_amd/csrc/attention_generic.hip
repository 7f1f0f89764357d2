// Attention over the paged cache, generic variants in float32 arithmetic.
//
// Cache layout (one K and one V pool per cache entry, pages of P = 64 tokens, the width
// of a wavefront): K [page][kv_head][P][head_dim] keeps a key's channels together, which
// is the order QK^T reduces over; V [page][kv_head][head_dim][P] keeps a channel's tokens
// together, which is the order PV reduces over. A token at position t of a sequence lives
// in page block_table[t / P] at offset t % P. (The reference's unwired paging primitive
// uses the same P and a page-major layout, native/src/paged_kv.h:48-83.)
#include "fw_common.h"
#include "fw_kernels.h"

#define ATTN_PAGE 64
#define ATTN_MAX_HEAD_DIM 1024      // of these plain kernels (the matrix-core kernels take up to 256)

// One wave per (row, head-vector). Head-vectors 0..nh-1 are queries, nh..nh+nkv-1 keys (head_dim
// channels each), the rest values (v_dim channels each, which may differ from head_dim). Per-head RMS norm then half-split rotation: channel i pairs with
// i + rotary_dim/2; out[i] = a cos - b sin, out[i + half] = b cos + a sin
// (native/include/flyweight_v2_native_kernels.hpp:1015-1050). Values are stored untouched.
template <typename TI, typename T>
__global__ __launch_bounds__(64) void qk_norm_rope_kv_write_kernel(
    const TI* __restrict__ qkv, T* __restrict__ q_out, const float* __restrict__ q_norm_weight,
    const float* __restrict__ k_norm_weight, float eps, const float* __restrict__ cos_table,
    const float* __restrict__ sin_table, int rotary_dim, T* __restrict__ k_pages, T* __restrict__ v_pages,
    const int32_t* __restrict__ block_table, int table_stride, const int32_t* __restrict__ row_seg,
    const int32_t* __restrict__ row_pos, int num_heads, int num_kv_heads, int head_dim, int v_dim, int interleaved, int width,
    const float* __restrict__ q_row_scale) {
    __shared__ float normed[ATTN_MAX_HEAD_DIM];
    const int row = blockIdx.x;
    const int vec = blockIdx.y;
    const int lane = threadIdx.x;
    const TI* source = qkv + (size_t)row * width + (vec < num_heads + num_kv_heads
                           ? (size_t)vec * head_dim
                           : (size_t)(num_heads + num_kv_heads) * head_dim + (size_t)(vec - num_heads - num_kv_heads) * v_dim);
    const int pos = row_pos[row];
    const int page = block_table[(size_t)row_seg[row] * table_stride + pos / ATTN_PAGE];
    const int slot = pos % ATTN_PAGE;

    if (vec >= num_heads + num_kv_heads) {      // value head: transposed store
        const int kvh = vec - num_heads - num_kv_heads;
        T* dest = v_pages + ((size_t)page * num_kv_heads + kvh) * v_dim * ATTN_PAGE;
        for (int d = lane; d < v_dim; d += 64) store_from_float(dest, (size_t)d * ATTN_PAGE + slot, load_as_float(source, d));
        return;
    }
    const bool is_query = vec < num_heads;
    const float* weight = is_query ? q_norm_weight : k_norm_weight;
    // a factor on the row's finished queries (one that depends on the row's position, say); keys take none
    const float factor = (is_query && q_row_scale) ? q_row_scale[row] : 1.0f;
    float inv = 1.0f;
    if (weight) {
        float sum = 0.0f;
        for (int d = lane; d < head_dim; d += 64) {
            const float v = load_as_float(source, d);
            sum += v * v;
        }
        sum = wave_sum(sum);
        inv = rsqrtf(sum / (float)head_dim + eps);
    }
    for (int d = lane; d < head_dim; d += 64) {
        const float v = load_as_float(source, d);
        normed[d] = weight ? v * inv * weight[d] : v;
    }
    __syncthreads();
    const int half = rotary_dim / 2;
    T* dest = is_query ? q_out + ((size_t)row * num_heads + vec) * head_dim
                       : k_pages + (((size_t)page * num_kv_heads + (vec - num_heads)) * ATTN_PAGE + slot) * head_dim;
    for (int d = lane; d < head_dim; d += 64) {
        float value = normed[d];
        if (d < rotary_dim) {
            // the pair's first channel turns as u cos - v sin, its second as v cos + u sin
            const bool is_first = interleaved ? (d & 1) == 0 : d < half;
            const int pair = interleaved ? d >> 1 : (d < half ? d : d - half);
            const float other = normed[interleaved ? d ^ 1 : (d < half ? d + half : d - half)];
            const float c = cos_table[(size_t)row * half + pair];
            const float s = sin_table[(size_t)row * half + pair];
            // one rounding of other * s, then one fused step: the same in every kernel that rotates
            value = fmaf(value, c, is_first ? -(other * s) : other * s);
        }
        store_from_float(dest, d, q_row_scale ? value * factor : value);
    }
}

// The same for heads of up to 64 channels (a channel per lane), eight rows of one head-vector per
// wave: what the wave reads for its eight rows is asked for together, so the chain of dependent
// loads in front (position and segment of the row, its page) is paid once for eight rows. A prompt
// of 2,048 rows has a hundred thousand (row, head-vector) pairs; as waves of one pair each they
// were bound by that chain. The rotation's partner channel comes from the partner lane. The same
// arithmetic in the same order as above.
#define QK_ROWS 8
template <typename TI, typename T>
__global__ __launch_bounds__(64) void qk_norm_rope_kv_write_rows_kernel(
    const TI* __restrict__ qkv, T* __restrict__ q_out, const float* __restrict__ q_norm_weight,
    const float* __restrict__ k_norm_weight, float eps, const float* __restrict__ cos_table,
    const float* __restrict__ sin_table, int rotary_dim, T* __restrict__ k_pages, T* __restrict__ v_pages,
    const int32_t* __restrict__ block_table, int table_stride, const int32_t* __restrict__ row_seg,
    const int32_t* __restrict__ row_pos, int num_heads, int num_kv_heads, int head_dim, int rows, int interleaved, int width,
    const float* __restrict__ q_row_scale) {
    const int r0 = blockIdx.x * QK_ROWS;
    const int vec = blockIdx.y;
    const int lane = threadIdx.x;
    const bool active = lane < head_dim;
    const bool is_value = vec >= num_heads + num_kv_heads, is_query = vec < num_heads;
    const float* weight = is_value ? nullptr : (is_query ? q_norm_weight : k_norm_weight);
    const int half = rotary_dim / 2;
    const bool turned = !is_value && lane < rotary_dim;
    const bool is_first = interleaved ? (lane & 1) == 0 : lane < half;
    const int pair = interleaved ? lane >> 1 : (lane < half ? lane : lane - half);
    const int partner = interleaved ? lane ^ 1 : (lane < half ? lane + half : lane - half);
    int row_of[QK_ROWS], pos[QK_ROWS], page[QK_ROWS];
    float v[QK_ROWS], c[QK_ROWS], sn[QK_ROWS];
#pragma unroll
    for (int i = 0; i < QK_ROWS; ++i) {
        row_of[i] = r0 + i < rows ? r0 + i : rows - 1;
        pos[i] = row_pos[row_of[i]];
        page[i] = row_seg[row_of[i]];
    }
#pragma unroll
    for (int i = 0; i < QK_ROWS; ++i) {
        v[i] = load_as_float(qkv + (size_t)row_of[i] * width + (size_t)vec * head_dim, active ? lane : 0);
        c[i] = turned ? cos_table[(size_t)row_of[i] * half + pair] : 1.0f;
        sn[i] = turned ? sin_table[(size_t)row_of[i] * half + pair] : 0.0f;
    }
    const float w = (weight && active) ? weight[lane] : 1.0f;
#pragma unroll
    for (int i = 0; i < QK_ROWS; ++i) page[i] = block_table[(size_t)page[i] * table_stride + pos[i] / ATTN_PAGE];
    if (is_value && sizeof(T) == 2) {
        // Eight rows that follow each other in one page, the first at a slot that is a multiple of eight (a
        // prompt portion that begins at such a position): a channel's eight values are 16 bytes side by side
        // in the transposed page and leave as one store instead of eight of 2 bytes.
        bool together = r0 + QK_ROWS <= rows && pos[0] % 8 == 0;
#pragma unroll
        for (int i = 1; i < QK_ROWS; ++i) together = together && page[i] == page[0] && pos[i] == pos[0] + i;
        if (together) {
            const int kvh = vec - num_heads - num_kv_heads;
            T* dest = v_pages + ((size_t)page[0] * num_kv_heads + kvh) * head_dim * ATTN_PAGE;
            uint32_t packed[QK_ROWS / 2];
#pragma unroll
            for (int i = 0; i < QK_ROWS / 2; ++i)
                packed[i] = (uint32_t)float_to_bf16_bits(v[2 * i]) | ((uint32_t)float_to_bf16_bits(v[2 * i + 1]) << 16);
            if (active) {
                uint32_t* to = reinterpret_cast<uint32_t*>(dest + (size_t)lane * ATTN_PAGE + pos[0] % ATTN_PAGE);
                typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;
                *reinterpret_cast<u32x4_t*>(to) = u32x4_t{packed[0], packed[1], packed[2], packed[3]};
            }
            return;
        }
    }
#pragma unroll
    for (int i = 0; i < QK_ROWS; ++i) {
        if (r0 + i >= rows) break;
        const int slot = pos[i] % ATTN_PAGE;
        if (is_value) {      // value head: transposed store
            const int kvh = vec - num_heads - num_kv_heads;
            T* dest = v_pages + ((size_t)page[i] * num_kv_heads + kvh) * head_dim * ATTN_PAGE;
            if (active) store_from_float(dest, (size_t)lane * ATTN_PAGE + slot, v[i]);
            continue;
        }
        float value = active ? v[i] : 0.0f;
        if (weight) {
            const float sum = wave_sum(value * value);
            const float inv = rsqrtf(sum / (float)head_dim + eps);
            value = value * inv * w;
        }
        const float other = __shfl(value, partner & 63, 64);
        if (lane < rotary_dim) value = fmaf(value, c[i], is_first ? -(other * sn[i]) : other * sn[i]);
        if (is_query && q_row_scale) value *= q_row_scale[row_of[i]];
        T* dest = is_query ? q_out + ((size_t)row_of[i] * num_heads + vec) * head_dim
                           : k_pages + (((size_t)page[i] * num_kv_heads + (vec - num_heads)) * ATTN_PAGE + slot) * head_dim;
        if (active) store_from_float(dest, lane, value);
    }
}

// The same once more for heads of 64 and 128 channels and values of whole 64s whose rows lie at 16 bytes: a lane holds four neighbouring channels, HEAD_LANES
// lanes a head, 64 / HEAD_LANES rows side by side, eight rows of a head-vector to a wave; a value's 64 channels a lane each, as above. With a channel a lane a
// wave's eight rows were eight sums over 64 lanes one behind the other, six trips through the LDS crossbar each, and every query waited for its row's
// position, segment and page, which keys and values alone need. What is left is the memory's: float32 sums in, bfloat16 out. 2,048 rows of 32 + 16 heads of 64
// 21.3 -> 13.1 us (2.9 TB/s), 801 rows 12.7 -> 8.2; 1,111 rows of 16 + 8 heads of 128 15.2 -> 10.3. The bits of one row to a wave: the squares
// are rounded and added in the order of the sum over a wave, channels 64 apart, then 32, 16, 8 and 4 over the lanes, 2 and 1 in the lane. (Eight rows one behind the other, as
// above, have a square fused with the first sum: float32 outputs that are normed were one unit in the last place away from those of fewer rows.)
template <typename TI> struct four_of { typedef float4 vector; };
template <> struct four_of<bf16_t> { typedef uint2 vector; };
__device__ __forceinline__ void four_floats(const float4 v, float (&x)[4]) { x[0] = v.x, x[1] = v.y, x[2] = v.z, x[3] = v.w; }
__device__ __forceinline__ void four_floats(const uint2 v, float (&x)[4]) {
    x[0] = bf16_bits_to_float(v.x & 0xffff), x[1] = bf16_bits_to_float(v.x >> 16);
    x[2] = bf16_bits_to_float(v.y & 0xffff), x[3] = bf16_bits_to_float(v.y >> 16);
}
__device__ __forceinline__ void store_four(float* to, const float (&x)[4]) { *reinterpret_cast<float4*>(to) = make_float4(x[0], x[1], x[2], x[3]); }
__device__ __forceinline__ void store_four(bf16_t* to, const float (&x)[4]) {
    *reinterpret_cast<uint2*>(to) = make_uint2((uint32_t)float_to_bf16_bits(x[0]) | ((uint32_t)float_to_bf16_bits(x[1]) << 16),
                                               (uint32_t)float_to_bf16_bits(x[2]) | ((uint32_t)float_to_bf16_bits(x[3]) << 16));
}
// the value of the lane N below in a row of 16 lanes, round its end
template <int N> __device__ __forceinline__ float turned_by(float v) { return __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(v), 0x120 + N, 0xF, 0xF, true)); }
template <typename TI, typename T, int HEAD_LANES>
__global__ __launch_bounds__(256) void qk_norm_rope_kv_write_wide_kernel(
    const TI* __restrict__ qkv, T* __restrict__ q_out, const float* __restrict__ q_norm_weight,
    const float* __restrict__ k_norm_weight, float eps, const float* __restrict__ cos_table,
    const float* __restrict__ sin_table, int rotary_dim, T* __restrict__ k_pages, T* __restrict__ v_pages,
    const int32_t* __restrict__ block_table, int table_stride, const int32_t* __restrict__ row_seg,
    const int32_t* __restrict__ row_pos, int num_heads, int num_kv_heads, int v_dim, int rows, int interleaved, int width,
    const float* __restrict__ q_row_scale, int units) {
    constexpr int D = 4 * HEAD_LANES, SIDE = 64 / HEAD_LANES, PASSES = QK_ROWS / SIDE;
    const int r0 = blockIdx.x * QK_ROWS, lane = threadIdx.x & 63;
    const int unit = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (unit >= units) return;
    if (unit >= num_heads + num_kv_heads) {     // 64 channels of a value head: transposed store
        const int blocks = v_dim / 64, kvh = (unit - num_heads - num_kv_heads) / blocks, d = (unit - num_heads - num_kv_heads) % blocks * 64 + lane;
        const size_t first = (size_t)(num_heads + num_kv_heads) * D + (size_t)kvh * v_dim + d;
        int pos[QK_ROWS], page[QK_ROWS];
        float v[QK_ROWS];
#pragma unroll
        for (int i = 0; i < QK_ROWS; ++i) {
            const int row = r0 + i < rows ? r0 + i : rows - 1;
            v[i] = load_as_float(qkv + (size_t)row * width, first);
            pos[i] = row_pos[row];
            page[i] = row_seg[row];
        }
#pragma unroll
        for (int i = 0; i < QK_ROWS; ++i) page[i] = block_table[(size_t)page[i] * table_stride + pos[i] / ATTN_PAGE];
        // eight rows that follow each other in one page leave as one store (see above)
        bool together = sizeof(T) == 2 && r0 + QK_ROWS <= rows && pos[0] % 8 == 0 && (uintptr_t)v_pages % 16 == 0;
#pragma unroll
        for (int i = 1; i < QK_ROWS; ++i) together = together && page[i] == page[0] && pos[i] == pos[0] + i;
        if (together) {
            uint32_t packed[QK_ROWS / 2];
#pragma unroll
            for (int i = 0; i < QK_ROWS / 2; ++i) packed[i] = (uint32_t)float_to_bf16_bits(v[2 * i]) | ((uint32_t)float_to_bf16_bits(v[2 * i + 1]) << 16);
            T* to = v_pages + (((size_t)page[0] * num_kv_heads + kvh) * v_dim + d) * ATTN_PAGE + pos[0] % ATTN_PAGE;
            *reinterpret_cast<uint4*>(to) = make_uint4(packed[0], packed[1], packed[2], packed[3]);
            return;
        }
#pragma unroll
        for (int i = 0; i < QK_ROWS; ++i)
            if (r0 + i < rows) store_from_float(v_pages, (((size_t)page[i] * num_kv_heads + kvh) * v_dim + d) * ATTN_PAGE + pos[i] % ATTN_PAGE, v[i]);
        return;
    }
    const bool is_query = unit < num_heads;
    const int own = lane % HEAD_LANES, half = rotary_dim / 2;      // this lane's channels are 4 own .. 4 own + 3
    const bool turned = 4 * own < rotary_dim;
    const bool is_first = 4 * own < half;                          // halves: the four channels are all in one of them
    const int pair = interleaved ? 2 * own : (is_first ? 4 * own : 4 * own - half);
    const float* weight = is_query ? q_norm_weight : k_norm_weight;
    int row_of[PASSES], pos[PASSES], page[PASSES];
    typename four_of<TI>::vector got[PASSES];
    float4 c[PASSES] = {}, s[PASSES] = {};
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
        const int row = r0 + i * SIDE + lane / HEAD_LANES;
        row_of[i] = row < rows ? row : rows - 1;
        if (!is_query) {                                            // asked for ahead of the rows: the page is another trip behind them
            pos[i] = row_pos[row_of[i]];
            page[i] = row_seg[row_of[i]];
        }
    }
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
        got[i] = *reinterpret_cast<const typename four_of<TI>::vector*>(qkv + (size_t)row_of[i] * width + (size_t)unit * D + 4 * own);
        if (turned) {
            const float *from_c = cos_table + (size_t)row_of[i] * half + pair, *from_s = sin_table + (size_t)row_of[i] * half + pair;
            if (interleaved) {
                const float2 two_c = *reinterpret_cast<const float2*>(from_c), two_s = *reinterpret_cast<const float2*>(from_s);
                c[i] = make_float4(two_c.x, two_c.x, two_c.y, two_c.y);
                s[i] = make_float4(-two_s.x, two_s.x, -two_s.y, two_s.y);
            } else {
                c[i] = *reinterpret_cast<const float4*>(from_c);
                const float4 four = *reinterpret_cast<const float4*>(from_s);
                s[i] = is_first ? make_float4(-four.x, -four.y, -four.z, -four.w) : four;
            }
        }
    }
    T* dest[PASSES];
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
        if (is_query) {
            dest[i] = q_out + ((size_t)row_of[i] * num_heads + unit) * D;
        } else {
            page[i] = block_table[(size_t)page[i] * table_stride + pos[i] / ATTN_PAGE];
            dest[i] = k_pages + (((size_t)page[i] * num_kv_heads + (unit - num_heads)) * ATTN_PAGE + pos[i] % ATTN_PAGE) * D;
        }
    }
    const float4 w4 = weight ? *reinterpret_cast<const float4*>(weight + 4 * own) : make_float4(1.f, 1.f, 1.f, 1.f);
    const int partner = (lane & ~(HEAD_LANES - 1)) | (turned ? (is_first ? own + half / 4 : own - half / 4) : own);
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
        float x[4];
        four_floats(got[i], x);
        if (weight) {
            float square[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) square[u] = fmaf(x[u], x[u], 0.0f);     // rounded: a plain product would be fused with the sum behind it
            if constexpr (HEAD_LANES == 32) {
                // the sum that a lane of a wave holds of its two channels: the second joins the first's square in one fused step
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    float low, high;
                    fw_quad_partners16(x[u], low, high);
                    square[u] = fmaf(high, high, low * low);
                }
            }
            // turned by 8, 4, 2 and 1 lanes, the sums of a step repeat at that distance: each is its partner's of a butterfly
#pragma unroll
            for (int u = 0; u < 4; ++u) square[u] += turned_by<8>(square[u]);
#pragma unroll
            for (int u = 0; u < 4; ++u) square[u] += turned_by<4>(square[u]);
#pragma unroll
            for (int u = 0; u < 4; ++u) square[u] += turned_by<2>(square[u]);
#pragma unroll
            for (int u = 0; u < 4; ++u) square[u] += turned_by<1>(square[u]);
            const float sum = (square[0] + square[2]) + (square[1] + square[3]);
            const float inv = rsqrtf(sum / (float)D + eps);
            x[0] = x[0] * inv * w4.x, x[1] = x[1] * inv * w4.y, x[2] = x[2] * inv * w4.z, x[3] = x[3] * inv * w4.w;
        }
        if (rotary_dim) {
            float other[4];
            if (interleaved) other[0] = x[1], other[1] = x[0], other[2] = x[3], other[3] = x[2];
            else if (half == 32)        // eight lanes on, of sixteen
#pragma unroll
                for (int u = 0; u < 4; ++u) other[u] = turned_by<8>(x[u]);
            else
#pragma unroll
                for (int u = 0; u < 4; ++u) other[u] = __shfl(x[u], partner, 64);
            if (turned) {
                x[0] = fmaf(x[0], c[i].x, other[0] * s[i].x), x[1] = fmaf(x[1], c[i].y, other[1] * s[i].y);
                x[2] = fmaf(x[2], c[i].z, other[2] * s[i].z), x[3] = fmaf(x[3], c[i].w, other[3] * s[i].w);
            }
        }
        if (is_query && q_row_scale) {
            const float factor = q_row_scale[row_of[i]];
#pragma unroll
            for (int u = 0; u < 4; ++u) x[u] *= factor;
        }
        if (r0 + i * SIDE + lane / HEAD_LANES < rows) store_four(dest[i] + 4 * own, x);
    }
}

extern "C" int fw_qk_norm_rope_kv_write(const void* qkv, int in_dtype, int row_stride, void* q_out, int dtype, const float* q_norm_weight,
                                        const float* k_norm_weight, float eps, const float* cos_table,
                                        const float* sin_table, int rotary_dim, void* k_pages, void* v_pages,
                                        const int32_t* block_table, int table_stride, const int32_t* row_seg,
                                        const int32_t* row_pos, int rows, int num_heads, int num_kv_heads,
                                        int head_dim, int v_dim, int page_size, int num_pages, int write_kv, int interleaved,
                                        int q_only, const float* q_row_scale, void* stream) {
    FW_REQUIRE(rows >= 0 && num_heads > 0 && num_kv_heads > 0, "qk_norm_rope: bad sizes rows=%d heads=%d kv_heads=%d", rows, num_heads, num_kv_heads);
    FW_REQUIRE(head_dim > 0 && head_dim <= ATTN_MAX_HEAD_DIM, "qk_norm_rope: head_dim %d outside 1..%d", head_dim, ATTN_MAX_HEAD_DIM);
    FW_REQUIRE(v_dim > 0 && v_dim <= ATTN_MAX_HEAD_DIM, "qk_norm_rope: value size %d outside 1..%d", v_dim, ATTN_MAX_HEAD_DIM);
    FW_REQUIRE(rotary_dim >= 0 && rotary_dim <= head_dim && rotary_dim % 2 == 0, "qk_norm_rope: rotary_dim %d must be even and at most head_dim %d", rotary_dim, head_dim);
    FW_REQUIRE(rotary_dim == 0 || (cos_table && sin_table), "qk_norm_rope: rotation asked for without tables");
    FW_REQUIRE(page_size == ATTN_PAGE, "qk_norm_rope: page size must be %d, got %d", ATTN_PAGE, page_size);
    FW_REQUIRE(num_pages > 0 && table_stride > 0, "qk_norm_rope: empty cache (pages=%d, table stride=%d)", num_pages, table_stride);
    FW_REQUIRE((q_norm_weight == nullptr) == (k_norm_weight == nullptr), "qk_norm_rope: q and k norm weights come together");
    FW_REQUIRE(rows <= 1 << 20, "qk_norm_rope: too many rows (%d)", rows);
    if (rows == 0) return 0;
    FW_REQUIRE(!(q_only && write_kv), "qk_norm_rope: rows that hold queries only bring no keys or values to store");
    const int vectors = write_kv ? num_heads + 2 * num_kv_heads : num_heads;
    const int needed = q_only ? num_heads * head_dim : (num_heads + num_kv_heads) * head_dim + num_kv_heads * v_dim;
    const int width = row_stride > 0 ? row_stride : needed;      // rows may hold more behind the values
    FW_REQUIRE(width >= needed, "qk_norm_rope: rows %d wide do not hold %d", width, needed);
    FW_REQUIRE(vectors <= 65535, "qk_norm_rope: too many heads (%d)", vectors);
    dim3 grid(rows, vectors);
    hipStream_t s = (hipStream_t)stream;
    // a prompt's rows, four channels to a lane, where 16 bytes of a row (8 in bfloat16) lie at such a place in everything that is read or stored so
    auto at = [](const void* p, int bytes) { return (uintptr_t)p % bytes == 0; };
    const int in_size = in_dtype == FW_F32 ? 4 : 2, out_size = dtype == FW_F32 ? 4 : 2;
    if ((head_dim == 64 || head_dim == 128) && v_dim % 64 == 0 && rows >= 8 * QK_ROWS && width % 4 == 0 && rotary_dim % 8 == 0 && at(qkv, 4 * in_size) &&
        at(q_out, 4 * out_size) && at(k_pages, 4 * out_size) && at(q_norm_weight, 16) && at(k_norm_weight, 16) && at(cos_table, 16) && at(sin_table, 16)) {
        const int units = write_kv ? num_heads + num_kv_heads + num_kv_heads * (v_dim / 64) : num_heads;
        dim3 wide((rows + QK_ROWS - 1) / QK_ROWS, (units + 3) / 4);
#define FW_QK_WIDE_LAUNCH(TI, T, LANES)                                                                              \
    qk_norm_rope_kv_write_wide_kernel<TI, T, LANES><<<wide, 256, 0, s>>>(                                            \
        (const TI*)qkv, (T*)q_out, q_norm_weight, k_norm_weight, eps, cos_table, sin_table, rotary_dim, (T*)k_pages, \
        (T*)v_pages, block_table, table_stride, row_seg, row_pos, num_heads, num_kv_heads, v_dim, rows, interleaved, width, q_row_scale, units)
#define FW_QK_WIDE(TI, T)                                \
    if (head_dim == 64) FW_QK_WIDE_LAUNCH(TI, T, 16);    \
    else FW_QK_WIDE_LAUNCH(TI, T, 32)
        if (in_dtype == FW_F32 && dtype == FW_F32) { FW_QK_WIDE(float, float); }
        else if (in_dtype == FW_F32 && dtype == FW_BF16) { FW_QK_WIDE(float, bf16_t); }
        else if (in_dtype == FW_BF16 && dtype == FW_BF16) { FW_QK_WIDE(bf16_t, bf16_t); }
        else FW_REQUIRE(false, "qk_norm_rope: unsupported dtypes in=%d out=%d", in_dtype, dtype);
#undef FW_QK_WIDE
#undef FW_QK_WIDE_LAUNCH
        FW_LAUNCH_CHECK("qk_norm_rope_kv_write");
        return 0;
    }
    if (head_dim <= 64 && v_dim == head_dim && rows >= 8 * QK_ROWS) {    // smaller heads, eight rows to a wave
        dim3 by_rows((rows + QK_ROWS - 1) / QK_ROWS, vectors);
#define FW_QK_ROWS_LAUNCH(TI, T)                                                                                     \
    qk_norm_rope_kv_write_rows_kernel<TI, T><<<by_rows, 64, 0, s>>>(                                                 \
        (const TI*)qkv, (T*)q_out, q_norm_weight, k_norm_weight, eps, cos_table, sin_table, rotary_dim, (T*)k_pages, \
        (T*)v_pages, block_table, table_stride, row_seg, row_pos, num_heads, num_kv_heads, head_dim, rows, interleaved, width, q_row_scale)
        if (in_dtype == FW_F32 && dtype == FW_F32) FW_QK_ROWS_LAUNCH(float, float);
        else if (in_dtype == FW_F32 && dtype == FW_BF16) FW_QK_ROWS_LAUNCH(float, bf16_t);
        else if (in_dtype == FW_BF16 && dtype == FW_BF16) FW_QK_ROWS_LAUNCH(bf16_t, bf16_t);
        else FW_REQUIRE(false, "qk_norm_rope: unsupported dtypes in=%d out=%d", in_dtype, dtype);
#undef FW_QK_ROWS_LAUNCH
        FW_LAUNCH_CHECK("qk_norm_rope_kv_write");
        return 0;
    }
#define FW_QK_LAUNCH(TI, T)                                                                                          \
    qk_norm_rope_kv_write_kernel<TI, T><<<grid, 64, 0, s>>>(                                                         \
        (const TI*)qkv, (T*)q_out, q_norm_weight, k_norm_weight, eps, cos_table, sin_table, rotary_dim, (T*)k_pages, \
        (T*)v_pages, block_table, table_stride, row_seg, row_pos, num_heads, num_kv_heads, head_dim, v_dim, interleaved, width, q_row_scale)
    if (in_dtype == FW_F32 && dtype == FW_F32) FW_QK_LAUNCH(float, float);
    else if (in_dtype == FW_F32 && dtype == FW_BF16) FW_QK_LAUNCH(float, bf16_t);
    else if (in_dtype == FW_BF16 && dtype == FW_BF16) FW_QK_LAUNCH(bf16_t, bf16_t);
    else FW_REQUIRE(false, "qk_norm_rope: unsupported dtypes in=%d out=%d", in_dtype, dtype);
#undef FW_QK_LAUNCH
    FW_LAUNCH_CHECK("qk_norm_rope_kv_write");
    return 0;
}

// One wave per (row, head). Keys are visited page by page, one key per lane; softmax is
// the running-maximum form in float32 (scores, maximum, exponentials, sum and the weighted
// sum of values all float32), as the reference's decode fallback computes it in two
// passes (native/include/flyweight_v2_qwen_kernels.hpp:12570-12585,12664-12704). The order
// of every sum depends only on the row's position and the window, never on the batch.
// A decode step has a wave per head and nothing beside it: its time is a chain of trips to memory, one page after the other.
// WIDE (float32, head sizes that are multiples of 4): keys and values come 16 bytes at a time, a page's first 64 value channels are
// asked for ahead of its scores. The same sums in the same order; 16 heads of 64
// channels, one row behind 301-308 keys 44 -> 20 us, 301 rows 161 -> 61 us.
template <typename T, bool WIDE>
__global__ __launch_bounds__(64) void attention_generic_kernel(
    const T* __restrict__ q, T* __restrict__ out, const T* __restrict__ k_pages, const T* __restrict__ v_pages,
    const int32_t* __restrict__ block_table, int table_stride, const int32_t* __restrict__ row_seg,
    const int32_t* __restrict__ row_pos, int num_heads, int num_kv_heads, int head_dim, int v_dim, float scale, int window,
    int chunk, float softcap, int keep_first, const float* __restrict__ sinks, const float* __restrict__ slopes) {
    __shared__ __attribute__((aligned(16))) float qs[ATTN_MAX_HEAD_DIM];
    __shared__ __attribute__((aligned(16))) float ps[ATTN_PAGE];
    const int row = blockIdx.x, head = blockIdx.y, lane = threadIdx.x;
    const int kvh = head / (num_heads / num_kv_heads);
    const int pos = row_pos[row];
    const int32_t* table = block_table + (size_t)row_seg[row] * table_stride;
    const T* query = q + ((size_t)row * num_heads + head) * head_dim;
    for (int d = lane; d < head_dim; d += 64) qs[d] = load_as_float(query, d);
    __syncthreads();
    const int first = fw_first_visible(pos, window, chunk);
    float running_max = -INFINITY, running_sum = 0.0f;
    float acc[ATTN_MAX_HEAD_DIM / 64] = {};
    // the pages of the kept first keys that lie before the first visible one, then those from it on
    const int kept = keep_first < first ? keep_first : first;              // keys 0 .. kept - 1 are seen beside first .. pos
    const int head_tiles = (kept + ATTN_PAGE - 1) / ATTN_PAGE < first / ATTN_PAGE ? (kept + ATTN_PAGE - 1) / ATTN_PAGE : first / ATTN_PAGE;
    const int tiles = head_tiles + pos / ATTN_PAGE - first / ATTN_PAGE + 1;
    for (int at = 0; at < tiles; ++at) {
        const int tile = at < head_tiles ? at : first / ATTN_PAGE + at - head_tiles;
        const int page = table[tile];
        const int t = tile * ATTN_PAGE + lane;
        const bool valid = (t >= first || t < kept) && t <= pos;
        float score = -INFINITY;
        // (a value's keys past the last one written hold anything: read, not used)
        float4 ahead[WIDE ? ATTN_PAGE / 4 : 1];
        if (WIDE) {
            const float4* value = reinterpret_cast<const float4*>(v_pages + (((size_t)page * num_kv_heads + kvh) * v_dim + (lane < v_dim ? lane : 0)) * ATTN_PAGE);
#pragma unroll
            for (int i = 0; i < ATTN_PAGE / 4; ++i) ahead[i] = value[i];
        }
        if (valid) {
            const T* key = k_pages + (((size_t)page * num_kv_heads + kvh) * ATTN_PAGE + lane) * head_dim;
            float dot = 0.0f;
            if (WIDE) {
                const float4* key4 = reinterpret_cast<const float4*>(key);
                const float4* q4 = reinterpret_cast<const float4*>(qs);
#pragma unroll 16
                for (int d = 0; d < head_dim / 4; ++d) {
                    const float4 k = key4[d], x = q4[d];
                    dot = fmaf(x.w, k.w, fmaf(x.z, k.z, fmaf(x.y, k.y, fmaf(x.x, k.x, dot))));
                }
            } else {
                for (int d = 0; d < head_dim; ++d) dot = fmaf(qs[d], load_as_float(key, d), dot);
            }
            score = dot * scale;
            if (softcap > 0.0f) score = softcap * tanhf(score / softcap);
            if (slopes) score -= slopes[head] * (float)(pos - t);      // a bias by distance, behind the cap
        }
        const float new_max = fmaxf(running_max, wave_max(score));
        const float p = valid ? expf(score - new_max) : 0.0f;
        const float alpha = expf(running_max - new_max);
        running_sum = running_sum * alpha + wave_sum(p);
        running_max = new_max;
        ps[lane] = p;
        __syncthreads();
        const int lo = (first - tile * ATTN_PAGE > 0 && kept <= tile * ATTN_PAGE) ? first - tile * ATTN_PAGE : 0;    // a masked key's weight is 0
        const int hi = pos - tile * ATTN_PAGE < ATTN_PAGE - 1 ? pos - tile * ATTN_PAGE : ATTN_PAGE - 1;
#pragma unroll
        for (int j = 0; j < ATTN_MAX_HEAD_DIM / 64; ++j) {
            const int d = lane + 64 * j;
            if (d < v_dim) {
                const T* value = v_pages + (((size_t)page * num_kv_heads + kvh) * v_dim + d) * ATTN_PAGE;
                float sum = 0.0f;
                if (WIDE) {
                    // a key outside lo .. hi has weight 0 and adds 0 times 0
                    const float4* value4 = reinterpret_cast<const float4*>(value);
                    const float4* p4 = reinterpret_cast<const float4*>(ps);
                    const bool whole = lo == 0 && hi == ATTN_PAGE - 1;
#pragma unroll
                    for (int i = 0; i < ATTN_PAGE / 4; ++i) {
                        float4 v = j == 0 ? ahead[i] : value4[i];
                        const float4 p = p4[i];
                        if (!whole) {
                            v.x = 4 * i >= lo && 4 * i <= hi ? v.x : 0.0f;
                            v.y = 4 * i + 1 >= lo && 4 * i + 1 <= hi ? v.y : 0.0f;
                            v.z = 4 * i + 2 >= lo && 4 * i + 2 <= hi ? v.z : 0.0f;
                            v.w = 4 * i + 3 >= lo && 4 * i + 3 <= hi ? v.w : 0.0f;
                        }
                        sum = fmaf(p.w, v.w, fmaf(p.z, v.z, fmaf(p.y, v.y, fmaf(p.x, v.x, sum))));
                    }
                } else {
                    for (int s = lo; s <= hi; ++s) sum = fmaf(ps[s], load_as_float(value, s), sum);
                }
                acc[j] = acc[j] * alpha + sum;
            }
        }
        __syncthreads();
    }
    float shrink = 1.0f;
    if (sinks) {        // one more term in the sum, with no value: exp(sink), not scaled
        const float sink = sinks[head];
        const float new_max = fmaxf(running_max, sink);
        shrink = expf(running_max - new_max);
        running_sum = running_sum * shrink + expf(sink - new_max);
    }
    T* dest = out + ((size_t)row * num_heads + head) * v_dim;
#pragma unroll
    for (int j = 0; j < ATTN_MAX_HEAD_DIM / 64; ++j) {
        const int d = lane + 64 * j;
        if (d < v_dim) store_from_float(dest, d, acc[j] * shrink / running_sum);
    }
}

// The same for steps of few rows, float32, head sizes that are multiples of 4: a workgroup of eight waves per (row, head), which take eight pages side by
// side. Scores, maxima, exponentials and a page's weighted sum are formed page by page as above, and the pages then folded in their order with the same
// expressions: bit for bit the same results. What it saves is the chain from page to page. us, a wave a row and head / eight pages, 16 heads in 8
// groups of 64 channels, one row of 20 / 64 / 100 / 300 / 1,100 / 3,000 keys 5.4 / 5.5, 4.8 / 5.5, 7.9 / 6.6, 15.5 / 10.1, 47.5 / 27.8, 136 / 67; sixteen
// rows 5.5 / 5.7, 5.0 / 5.7, 8.1 / 6.8, 17.9 / 11.0, 54.9 / 29.7, 161 / 75; 8 heads of 96 channels, 32 rows of 64 / 300 / 3,000 keys 7.4 / 7.8, 28.1 / 17.1,
// 266 / 138; 4 heads of 256, 64 rows 10.3 / 9.2, 56.1 / 29.4, 586 / 252. A context of one page has nothing to take side by side and costs up to 0.8 us
// more, with narrow heads; how long contexts are the caller of a recorded step does not know. With rows times heads
// enough to fill the chip the waves above have no idle compute units beside them.
#define SIDE 8
#define PAGES_MOST 256          // rows times heads: a workgroup a compute unit
__global__ __launch_bounds__(64 * SIDE) void attention_pages_kernel(
    const float* __restrict__ q, float* __restrict__ out, const float* __restrict__ k_pages, const float* __restrict__ v_pages,
    const int32_t* __restrict__ block_table, int table_stride, const int32_t* __restrict__ row_seg,
    const int32_t* __restrict__ row_pos, int num_heads, int num_kv_heads, int head_dim, int v_dim, float scale, int window,
    int chunk, float softcap, int keep_first, const float* __restrict__ sinks, const float* __restrict__ slopes) {
    __shared__ __attribute__((aligned(16))) float qs[ATTN_MAX_HEAD_DIM];
    __shared__ __attribute__((aligned(16))) float ps[SIDE][ATTN_PAGE];
    __shared__ float page_max[SIDE], page_sum[SIDE], parts[SIDE][64 * SIDE];
    const int row = blockIdx.x, head = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kvh = head / (num_heads / num_kv_heads);
    const int pos = row_pos[row];
    const int32_t* table = block_table + (size_t)row_seg[row] * table_stride;
    const float* query = q + ((size_t)row * num_heads + head) * head_dim;
    for (int d = tid; d < head_dim; d += 64 * SIDE) qs[d] = query[d];
    const int first = fw_first_visible(pos, window, chunk);
    const int kept = keep_first < first ? keep_first : first;
    const int head_tiles = (kept + ATTN_PAGE - 1) / ATTN_PAGE < first / ATTN_PAGE ? (kept + ATTN_PAGE - 1) / ATTN_PAGE : first / ATTN_PAGE;
    const int tiles = head_tiles + pos / ATTN_PAGE - first / ATTN_PAGE + 1;
    float running_max = -INFINITY, running_sum = 0.0f, acc = 0.0f;         // acc: channel tid
    for (int at0 = 0; at0 < tiles; at0 += SIDE) {
        const int here = tiles - at0 < SIDE ? tiles - at0 : SIDE;
        const bool busy = wave < here;
        const int at = at0 + (busy ? wave : 0);
        const int tile = at < head_tiles ? at : first / ATTN_PAGE + at - head_tiles;
        const int page = table[tile];
        const int t = tile * ATTN_PAGE + lane;
        const bool valid = busy && (t >= first || t < kept) && t <= pos;
        const float* values = v_pages + ((size_t)page * num_kv_heads + kvh) * v_dim * ATTN_PAGE;
        float4 ahead[ATTN_PAGE / 4];
        const float4* value_ahead = reinterpret_cast<const float4*>(values + (size_t)(lane < v_dim ? lane : 0) * ATTN_PAGE);
        // (a load of 64 rows' pieces costs the compute unit 64 lookups: a wave without a page asks for nothing)
        if (busy)
#pragma unroll
            for (int i = 0; i < ATTN_PAGE / 4; ++i) ahead[i] = value_ahead[i];
        fw_lds_barrier();                                                   // the query is there; the parts before have been folded (the loads stay on their way)
        float score = -INFINITY;
        if (valid) {
            const float4* key4 = reinterpret_cast<const float4*>(k_pages + (((size_t)page * num_kv_heads + kvh) * ATTN_PAGE + lane) * head_dim);
            const float4* q4 = reinterpret_cast<const float4*>(qs);
            float dot = 0.0f;
#pragma unroll 16
            for (int d = 0; d < head_dim / 4; ++d) {
                const float4 k = key4[d], x = q4[d];
                dot = fmaf(x.w, k.w, fmaf(x.z, k.z, fmaf(x.y, k.y, fmaf(x.x, k.x, dot))));
            }
            score = dot * scale;
            if (softcap > 0.0f) score = softcap * tanhf(score / softcap);
            if (slopes) score -= slopes[head] * (float)(pos - t);
        }
        const float most = wave_max(score);
        if (busy && lane == 0) page_max[wave] = most;
        fw_lds_barrier();
        if (busy) {
            float new_max = running_max;
            for (int i = 0; i <= wave; ++i) new_max = fmaxf(new_max, page_max[i]);
            const float p = valid ? expf(score - new_max) : 0.0f;
            const float sum = wave_sum(p);
            if (lane == 0) page_sum[wave] = sum;
            ps[wave][lane] = p;
            const int lo = (first - tile * ATTN_PAGE > 0 && kept <= tile * ATTN_PAGE) ? first - tile * ATTN_PAGE : 0;
            const int hi = pos - tile * ATTN_PAGE < ATTN_PAGE - 1 ? pos - tile * ATTN_PAGE : ATTN_PAGE - 1;
            const bool whole = lo == 0 && hi == ATTN_PAGE - 1;
            const float4* p4 = reinterpret_cast<const float4*>(ps[wave]);   // (a wave's own: its writes are ahead of its reads)
            for (int j = 0; 64 * j < v_dim; ++j) {
                const int d = lane + 64 * j;
                if (d < v_dim) {
                    const float4* value4 = reinterpret_cast<const float4*>(values + (size_t)d * ATTN_PAGE);
                    float part = 0.0f;
#pragma unroll
                    for (int i = 0; i < ATTN_PAGE / 4; ++i) {
                        float4 v = j == 0 ? ahead[i] : value4[i];
                        const float4 w = p4[i];
                        if (!whole) {
                            v.x = 4 * i >= lo && 4 * i <= hi ? v.x : 0.0f;
                            v.y = 4 * i + 1 >= lo && 4 * i + 1 <= hi ? v.y : 0.0f;
                            v.z = 4 * i + 2 >= lo && 4 * i + 2 <= hi ? v.z : 0.0f;
                            v.w = 4 * i + 3 >= lo && 4 * i + 3 <= hi ? v.w : 0.0f;
                        }
                        part = fmaf(w.w, v.w, fmaf(w.z, v.z, fmaf(w.y, v.y, fmaf(w.x, v.x, part))));
                    }
                    parts[wave][d] = part;
                }
            }
        }
        fw_lds_barrier();
        for (int i = 0; i < here; ++i) {
            const float new_max = fmaxf(running_max, page_max[i]);
            const float alpha = expf(running_max - new_max);
            running_sum = running_sum * alpha + page_sum[i];
            running_max = new_max;
            if (tid < v_dim) acc = acc * alpha + parts[i][tid];
        }
    }
    float shrink = 1.0f;
    if (sinks) {
        const float sink = sinks[head];
        const float new_max = fmaxf(running_max, sink);
        shrink = expf(running_max - new_max);
        running_sum = running_sum * shrink + expf(sink - new_max);
    }
    if (tid < v_dim) out[((size_t)row * num_heads + head) * v_dim + tid] = acc * shrink / running_sum;
}

extern "C" int fw_attention_generic(const void* q, void* out, int dtype, const void* k_pages,
                                    const void* v_pages, const int32_t* block_table, int table_stride,
                                    const int32_t* row_seg, const int32_t* row_pos, int rows, int num_heads,
                                    int num_kv_heads, int head_dim, int v_dim, float scale, int window, int chunk,
                                    float softcap, int keep_first, const float* sinks, const float* slopes, int page_size, int num_pages, void* stream) {
    FW_REQUIRE(chunk >= 0 && softcap >= 0.0f, "attention: chunk %d and soft cap %g must not be negative", chunk, (double)softcap);
    FW_REQUIRE(keep_first >= 0 && (keep_first == 0 || chunk == 0), "attention: %d first keys are kept beside a window, not beside chunks", keep_first);
    FW_REQUIRE(rows >= 0 && num_heads > 0 && num_kv_heads > 0 && num_heads % num_kv_heads == 0,
               "attention: heads %d must be a positive multiple of kv heads %d", num_heads, num_kv_heads);
    FW_REQUIRE(head_dim > 0 && head_dim <= ATTN_MAX_HEAD_DIM, "attention: head_dim %d outside 1..%d", head_dim, ATTN_MAX_HEAD_DIM);
    FW_REQUIRE(v_dim > 0 && v_dim <= ATTN_MAX_HEAD_DIM, "attention: value size %d outside 1..%d", v_dim, ATTN_MAX_HEAD_DIM);
    FW_REQUIRE(page_size == ATTN_PAGE, "attention: page size must be %d, got %d", ATTN_PAGE, page_size);
    FW_REQUIRE(window >= 0, "attention: window must be 0 (all keys) or positive, got %d", window);
    FW_REQUIRE(num_pages > 0 && table_stride > 0, "attention: empty cache (pages=%d, table stride=%d)", num_pages, table_stride);
    FW_REQUIRE(rows <= 1 << 20 && num_heads <= 65535, "attention: too many rows/heads (%d, %d)", rows, num_heads);
    if (rows == 0) return 0;
    dim3 grid(rows, num_heads);
#define FW_ATTENTION_LAUNCH(T, WIDE)                                                                                              \
    attention_generic_kernel<T, WIDE><<<grid, 64, 0, (hipStream_t)stream>>>(                                                      \
        (const T*)q, (T*)out, (const T*)k_pages, (const T*)v_pages, block_table, table_stride, row_seg, row_pos, num_heads,       \
        num_kv_heads, head_dim, v_dim, scale, window, chunk, softcap, keep_first, sinks, slopes)
    const bool wide = dtype == FW_F32 && head_dim % 4 == 0 && ((uintptr_t)k_pages | (uintptr_t)v_pages) % 16 == 0;
    if (wide && v_dim <= 64 * SIDE && (long long)rows * num_heads <= PAGES_MOST)          // (a thread has a channel of the output)
        attention_pages_kernel<<<grid, 64 * SIDE, 0, (hipStream_t)stream>>>(
            (const float*)q, (float*)out, (const float*)k_pages, (const float*)v_pages, block_table, table_stride, row_seg, row_pos, num_heads, num_kv_heads,
            head_dim, v_dim, scale, window, chunk, softcap, keep_first, sinks, slopes);
    else if (wide) FW_ATTENTION_LAUNCH(float, true);
    else if (dtype == FW_F32) FW_ATTENTION_LAUNCH(float, false);
    else if (dtype == FW_BF16) FW_ATTENTION_LAUNCH(bf16_t, false);
#undef FW_ATTENTION_LAUNCH
    else
        FW_REQUIRE(false, "attention: unknown dtype %d", dtype);
    FW_LAUNCH_CHECK("attention_generic");
    return 0;
}
