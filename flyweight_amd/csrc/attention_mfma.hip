// Attention over the paged cache on the matrix cores (bfloat16 cache, float32 softmax).
//
// One wave works on 16 "columns" against the keys of one kv head. For a prompt portion a
// column is a query row (16 consecutive rows of one segment and one head per wave, four such
// waves per workgroup sharing the pages through LDS). For decode
// a column is one of the query heads that share the kv head, and the keys are split between
// workgroups in runs of SPLIT_PAGES pages whose partial results (running maximum, sum and
// unnormalised output) the workgroup that finishes last merges in the order of the keys.
//
// The products are formed transposed so that nothing has to change lanes between them:
//   S^T[key][col] = K[key][d] . Q^T[d][col]        (v_mfma_f32_16x16x32_bf16, k = d)
//   O^T[d][col]  += V^T[d][key] . P^T[key][col]    (k = key)
// Lane (col, g) receives the scores of keys 4g..4g+3 of each 16-key tile, which is exactly
// what it must supply as P^T for keys {4g..4g+3} of two tiles if the 32 keys of the second
// product are taken in that order; V^T is fetched in the same order, which its layout
// ([page][kv_head][head_dim][64 keys]: a channel's keys together) makes two 8-byte loads.
// K ([page][kv_head][64 keys][head_dim]) is fetched straight into operand registers too.
// Maximum, exponentials, sums and the rescaling of O are float32; P is rounded to bfloat16
// for the second product. The reference's fast decode tier has the same split-and-merge shape
// (native/src/split_kv.h:77-124, native/src/v2_runtime.cpp:24241-24267).
#include "fw_common.h"
#include "fw_kernels.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;

#define PAGE 64
#define SPLIT_PAGES 4           // keys per decode split = 256, whatever the batch
#define NEG_BIG (-1.0e30f)
#define PART_STRIDE(head_dim) ((head_dim) + 4)   // unnormalised output, maximum, sum, two unused: rows stay 16-byte aligned

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    return (uint32_t)float_to_bf16_bits(lo) | ((uint32_t)float_to_bf16_bits(hi) << 16);
}
// the same in one instruction (v_cvt_pk_bf16_f32, round to nearest even)
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
__device__ __forceinline__ uint32_t pack_bf16_pair(float lo, float hi) {
    const f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// State of one wave: 16 columns, HD channels (HD a multiple of 32 that holds both a key's head_dim
// channels and a value's v_dim channels, which may differ; query channels >= head_dim are zero, output
// channels >= v_dim are computed from the last real one and never stored).
template <int HD>
struct Columns {
    bf16x8 q[HD / 32];          // this lane's part of Q^T: column lane % 16, d = 32 c + 8 (lane / 16) ..
    f32x4 o[HD / 16];           // O^T: column lane % 16, d = 16 t + 4 (lane / 16) + r
    float m, l;                 // running maximum (in units of log2) and this lane's share of the sum
};

// One page of 64 keys against NH sets of columns that share the keys (query heads of one kv
// group over the same rows): the keys and values are read once for all of them. `lo`/`hi`: the
// keys of this page that this lane's column may see are those with lo <= key <= hi
// (page-relative; hi < 0: none), and with `kept` > 0 also the keys below `kept`. `last_written`: keys beyond it hold whatever an earlier owner of
// the page left, and are zeroed before they meet P = 0: here if CLEAN_V, else the caller has done
// it (the prompt kernel does when it copies a page to LDS). K_PADDED: a key's row holds HD channels,
// those past head_dim zero (the prompt kernel's LDS tile), so every lane loads; else the lanes past
// head_dim take zeros without loading.
//
// The softmax arithmetic (one exponential per score on the quarter-rate unit) takes more issue
// cycles than the matrix products take on their pipe, so the work is laid out in phases, each
// over all heads, with one short branch (the mask) that touches nothing but the scores: the
// compiler can then let the products of one head run behind the arithmetic of another, and the
// accumulators stay where they are (a join of two paths that both write them costs a register
// move per accumulator and page). A page of which every key counts for every column of the wave
// (all pages but those on the diagonal, at a window's edge, and a sequence's last) skips the
// mask. The scale is folded into the exponent's argument: the maximum is taken over the raw
// scores (the scale is positive) and kept scaled.
template <int HD, int NH, bool CLEAN_V, bool K_PADDED>
__device__ __forceinline__ void attend_page(Columns<HD> (&c)[NH], const uint16_t* __restrict__ k_page,
                                            const uint16_t* __restrict__ v_page, int head_dim, int v_dim, float scale_log2,
                                            int lo, int hi, int last_written, int k_stride, int v_stride,
                                            float cap = 0.0f, float cap_scale = 0.0f, int kept = 0, const float* dist = nullptr) {
    const int lane = threadIdx.x & 63;
    const int i16 = lane & 15, g = lane >> 4;
    // all key loads of the page are issued before the first product
    bf16x8 kf[4][HD / 32];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
        const uint16_t* key = k_page + (size_t)(kt * 16 + i16) * k_stride + g * 8;
#pragma unroll
        for (int dc = 0; dc < HD / 32; ++dc) {
            if (K_PADDED) {
                kf[kt][dc] = *reinterpret_cast<const bf16x8*>(key + dc * 32);
            } else {
                kf[kt][dc] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
                if (dc * 32 + g * 8 < head_dim) kf[kt][dc] = *reinterpret_cast<const bf16x8*>(key + dc * 32);
            }
        }
    }
    // scores of all heads
    f32x4 s[NH][4];
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            s[h][kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int dc = 0; dc < HD / 32; ++dc)
                s[h][kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[kt][dc], c[h].q[dc], s[h][kt], 0, 0, 0);
        }
    // A soft cap on the scores: s <- cap * tanh(s * scale / cap) (cap_scale = scale / cap; the caller then
    // passes log2(e) as the exponent's scale). tanh(x) = 1 - 2 / (1 + e^2x): exact at both ends, where
    // e^2x is 0 or infinite; the hardware's 2^x and reciprocal leave the scores to about 1e-6 of the cap.
    if (cap > 0.0f) {
        const float twice = 2.0f * cap_scale * 1.4426950408889634f;
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
            for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float e = __builtin_amdgcn_exp2f(s[h][kt][r] * twice);
                    s[h][kt][r] = cap - 2.0f * cap * __builtin_amdgcn_rcpf(1.0f + e);
                }
    }
    // A bias by distance, behind the cap: dist[h] (this lane's column of head set h; null: none) times the
    // number of keys between the column's own position (`hi`, page-relative) and the key is taken off, in
    // the units of the raw scores.
    if (dist) {
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
            for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                for (int r = 0; r < 4; ++r) s[h][kt][r] = fmaf(-dist[h], (float)(hi - (kt * 16 + g * 4 + r)), s[h][kt][r]);
    }
    // `kept`: the keys below it (page-relative; <= 0: none) are seen as well, whatever `lo` says
    const bool full = __all((lo <= 0 || kept >= lo) && hi >= PAGE - 1) && last_written >= PAGE - 1;
    if (!full) {
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int key = kt * 16 + g * 4 + r;
                const bool seen = (key >= lo || key < kept) && key <= hi;
#pragma unroll
                for (int h = 0; h < NH; ++h) s[h][kt][r] = seen ? s[h][kt][r] : NEG_BIG;
            }
    }
    // the running maximum of each column: over this lane's 16 scores, then over the four lanes
    // that share the column
    float alpha[NH], shift[NH];
    bool rose = false;
#pragma unroll
    for (int h = 0; h < NH; ++h) {
        float page_max = NEG_BIG;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) page_max = fmaxf(page_max, s[h][kt][r]);
        page_max = fw_quad_max(page_max);
        // a column that has seen no key yet keeps NEG_BIG (the raw maximum times the scale would overflow)
        const bool any_key = page_max > 0.5f * NEG_BIG;
        const float new_max = fmaxf(c[h].m, any_key ? page_max * scale_log2 : NEG_BIG);
        // the hardware's 2^x: arguments are <= 0 here, and one far below (a first page, a masked key
        // against a real maximum) gives 0
        alpha[h] = __builtin_amdgcn_exp2f(c[h].m - new_max);
        rose |= alpha[h] != 1.0f;
        c[h].m = new_max;
        // a masked score (NEG_BIG) times the scale is far below any maximum: its exponential is 0.
        // A column without any key so far (maximum NEG_BIG) subtracts nothing, so that the same holds.
        shift[h] = new_max > 0.5f * NEG_BIG ? -new_max : 0.0f;
    }
    // One head of up to 64 channels whose output lies in ordinary registers: rescaling it always
    // (sixteen multiplications by a factor that is 1 after the first pages) costs less than the
    // register moves that joining two paths, of which one writes the output, costs per page.
    if (NH == 1 && HD <= 64) {
#pragma unroll
        for (int t = 0; t < HD / 16; ++t) c[0].o[t] *= alpha[0];
    } else if (__any(rose)) {   // the maximum of some column rose (seldom after the first pages)
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
            for (int t = 0; t < HD / 16; ++t) c[h].o[t] *= alpha[h];
    }
    uint32_t p[NH][4][2];
#pragma unroll
    for (int h = 0; h < NH; ++h) {
        float sum = 0.0f;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            float e[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                e[r] = __builtin_amdgcn_exp2f(fmaf(s[h][kt][r], scale_log2, shift[h]));
                sum += e[r];
            }
            p[h][kt][0] = pack_bf16_pair(e[0], e[1]);
            p[h][kt][1] = pack_bf16_pair(e[2], e[3]);
        }
        c[h].l = c[h].l * alpha[h] + sum;
    }
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
        bf16x8 pf[NH];
#pragma unroll
        for (int h = 0; h < NH; ++h) {
            u32x4 pw = {p[h][2 * kb][0], p[h][2 * kb][1], p[h][2 * kb + 1][0], p[h][2 * kb + 1][1]};
            pf[h] = __builtin_bit_cast(bf16x8, pw);
        }
        const int key_a = kb * 32 + g * 4, key_b = key_a + 16;
        // keys <= last_written are kept: two keys per 32-bit word, the low half first. Without branches:
        // one between the load of V and the product would put every product into a block of its own.
        auto kept = [&](int first_key) -> uint32_t {
            return first_key + 1 <= last_written ? 0xffffffffu : (first_key <= last_written ? 0xffffu : 0u);
        };
        const uint32_t keep_a0 = kept(key_a), keep_a1 = kept(key_a + 2), keep_b0 = kept(key_b), keep_b1 = kept(key_b + 2);
        // Every channel tile of the template is computed, those past head_dim from the last real
        // channel again (their output is never stored): a branch around a matrix product whose
        // result is read right behind the branch is not safe. The compiler spaces a product and
        // the first read of its result inside one block, but where the read was the target of
        // a taken branch it came one instruction after the product and saw the registers that
        // the product writes last still unwritten (head sizes below the template's, two of four
        // components stale).
#pragma unroll
        for (int t = 0; t < HD / 16; ++t) {
            const int channel = t * 16 + i16 < v_dim ? t * 16 + i16 : v_dim - 1;
            const uint16_t* value = v_page + (size_t)channel * v_stride;
            const u32x2 va = *reinterpret_cast<const u32x2*>(value + key_a), vb = *reinterpret_cast<const u32x2*>(value + key_b);
            u32x4 vw = {va[0], va[1], vb[0], vb[1]};
            if (CLEAN_V) vw = u32x4{va[0] & keep_a0, va[1] & keep_a1, vb[0] & keep_b0, vb[1] & keep_b1};
            const bf16x8 vf = __builtin_bit_cast(bf16x8, vw);
#pragma unroll
            for (int h = 0; h < NH; ++h) c[h].o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[h], c[h].o[t], 0, 0, 0);
        }
    }
    // for the same reason the last products have left the pipe before control leaves this function
    fw_mfma_drain();
}

// ---- pages that stream through registers (decode, up to 128 channels) ---------------------------
// The keys and values of a page on their way into a wave's registers. A matrix product sums over its
// operands in any order, so the key that stands in row i of score tile kt is chosen to suit the values: 32 (kt / 2)
// + 8 (i / 4) + 4 (kt % 2) + i % 4. Then the eight keys whose probabilities a lane holds for half a page
// follow one another, and their values are one load of 16 bytes (four lanes together 64 bytes of a channel).
template <int HD>
struct PageOnWay {
    u32x4 k[4][HD / 32], v[2][HD / 16];
};
// Every lane's byte offsets in a page. Loads go through a buffer descriptor that ends with the page: channels past
// head_dim or v_dim give zeros, and a page that is not wanted has a descriptor of no bytes and costs no traffic.
template <int HD>
struct PageOffsets {
    uint32_t k[4][HD / 32], v;
    __device__ __forceinline__ PageOffsets(int head_dim) {
        const int lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int dc = 0; dc < HD / 32; ++dc) {
                const int key = (kt >> 1) * 32 + (i16 >> 2) * 8 + (kt & 1) * 4 + (i16 & 3), channel = dc * 32 + g * 8;
                k[kt][dc] = channel < head_dim ? (uint32_t)(key * head_dim + channel) * 2 : 0x7ffffff0u;
            }
        v = (uint32_t)(i16 * PAGE + g * 8) * 2;
    }
};
__device__ __forceinline__ u32x4 page_words(fw_buffer from, uint32_t at) { return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(from, at, 0, 0)); }
template <int HD>
__device__ __forceinline__ void ask_for_keys(PageOnWay<HD>& page, const PageOffsets<HD>& at, fw_buffer from) {
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int dc = 0; dc < HD / 32; ++dc) page.k[kt][dc] = page_words(from, at.k[kt][dc]);
}
template <int HD>
__device__ __forceinline__ void ask_for_values(PageOnWay<HD>& page, const PageOffsets<HD>& at, fw_buffer from) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int t = 0; t < HD / 16; ++t) page.v[kb][t] = page_words(from, at.v + t * 16 * PAGE * 2 + kb * 64);
}

// One page against one set of columns, as attend_page takes it: the same scores, maxima and exponentials, summed in the
// order of PageOnWay. As soon as the keys (values) have met their products, `ask_keys` (`ask_values`) asks for those of
// a later page into the same registers, so that the wave's loads never pause.
template <int HD, typename AskKeys, typename AskValues>
__device__ __forceinline__ void attend_on_way(Columns<HD>& c, PageOnWay<HD>& page, float scale_log2, int lo, int hi, float cap, float cap_scale, int kept,
                                              bool biased, float dist, AskKeys ask_keys, AskValues ask_values) {
    const int g = (threadIdx.x & 63) >> 4;
    f32x4 s[4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
        s[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int dc = 0; dc < HD / 32; ++dc)
            s[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, page.k[kt][dc]), c.q[dc], s[kt], 0, 0, 0);
    }
    fw_mfma_drain();        // the branches below read the scores
    ask_keys();
    // this lane's score [kt][r] is that of key 32 (kt / 2) + 8 g + 4 (kt % 2) + r
    auto key_of = [&](int kt, int r) { return (kt >> 1) * 32 + g * 8 + (kt & 1) * 4 + r; };
    if (cap > 0.0f) {
        const float twice = 2.0f * cap_scale * 1.4426950408889634f;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float e = __builtin_amdgcn_exp2f(s[kt][r] * twice);
                s[kt][r] = cap - 2.0f * cap * __builtin_amdgcn_rcpf(1.0f + e);
            }
    }
    if (biased) {
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) s[kt][r] = fmaf(-dist, (float)(hi - key_of(kt, r)), s[kt][r]);
    }
    // a page with keys that do not count: their scores leave the sum, and the values behind the row's own
    // position (an earlier owner's, perhaps no numbers) are cleared before they meet a probability of 0
    if (hi < PAGE - 1 || !(lo <= 0 || kept >= lo)) {
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int key = key_of(kt, r);
                s[kt][r] = (key >= lo || key < kept) && key <= hi ? s[kt][r] : NEG_BIG;
            }
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const int key = kb * 32 + g * 8 + 2 * w;
                const uint32_t keep = key + 1 <= hi ? 0xffffffffu : (key <= hi ? 0xffffu : 0u);
#pragma unroll
                for (int t = 0; t < HD / 16; ++t) page.v[kb][t][w] &= keep;
            }
    }
    float page_max = NEG_BIG;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) page_max = fmaxf(page_max, s[kt][r]);
    page_max = fw_quad_max(page_max);
    // a column that has seen no key yet keeps NEG_BIG and subtracts nothing (attend_page)
    const float new_max = fmaxf(c.m, page_max > 0.5f * NEG_BIG ? page_max * scale_log2 : NEG_BIG);
    const float alpha = __builtin_amdgcn_exp2f(c.m - new_max);
    const float shift = new_max > 0.5f * NEG_BIG ? -new_max : 0.0f;
    c.m = new_max;
#pragma unroll
    for (int t = 0; t < HD / 16; ++t) c.o[t] *= alpha;
    u32x4 p[2];
    float sum = 0.0f;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
        float e[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            e[r] = __builtin_amdgcn_exp2f(fmaf(s[kt][r], scale_log2, shift));
            sum += e[r];
        }
        p[kt >> 1][(kt & 1) * 2] = pack_bf16_pair(e[0], e[1]);
        p[kt >> 1][(kt & 1) * 2 + 1] = pack_bf16_pair(e[2], e[3]);
    }
    c.l = c.l * alpha + sum;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int t = 0; t < HD / 16; ++t)
            c.o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, page.v[kb][t]), __builtin_bit_cast(bf16x8, p[kb]), c.o[t], 0, 0, 0);
    fw_mfma_drain();        // before control leaves (attend_page)
    ask_values();
}

// The second of two halves that shared a tile's pages out leaves its maximum, sum and output to the same lane of the first, which joins them with its own.
template <int HD, int NH>
__device__ __forceinline__ void leave_columns(const Columns<HD> (&c)[NH], float* left) {        // left: [NH][HD / 4 + 2][256], this thread's place
    constexpr int VALUES = HD / 4 + 2;
#pragma unroll
    for (int h = 0; h < NH; ++h) {
        left[(h * VALUES + HD / 4) * 256] = c[h].m;
        left[(h * VALUES + HD / 4 + 1) * 256] = c[h].l;
#pragma unroll
        for (int t = 0; t < HD / 16; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) left[(h * VALUES + t * 4 + r) * 256] = c[h].o[t][r];
    }
}
template <int HD, int NH>
__device__ __forceinline__ void join_columns(Columns<HD> (&c)[NH], const float* left) {
    constexpr int VALUES = HD / 4 + 2;
#pragma unroll
    for (int h = 0; h < NH; ++h) {
        const float other = left[(h * VALUES + HD / 4) * 256], top = fmaxf(c[h].m, other);
        // (a half without any key of this row keeps NEG_BIG: its factor is 0)
        const float mine = __builtin_amdgcn_exp2f(c[h].m - top), theirs = __builtin_amdgcn_exp2f(other - top);
        c[h].m = top;
        c[h].l = c[h].l * mine + left[(h * VALUES + HD / 4 + 1) * 256] * theirs;
#pragma unroll
        for (int t = 0; t < HD / 16; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) c[h].o[t][r] = c[h].o[t][r] * mine + left[(h * VALUES + t * 4 + r) * 256] * theirs;
    }
}

// The output of a lane's row for the first `heads` of its columns' heads, `v_dim` channels each from `dest` on; sinks: of those heads, or null
template <int HD, int NH>
__device__ __forceinline__ void store_columns(const Columns<HD> (&c)[NH], bool valid, int heads, const float* __restrict__ sinks, uint16_t* __restrict__ dest, int v_dim) {
    const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int h = 0; h < NH; ++h) {
        float l = fw_quad_sum(c[h].l);
        if (!valid || h >= heads) continue;
        float inv = 1.0f / l;
        if (sinks) {        // one more term in the sum, with no value: exp(sink), not scaled
            const float sink = sinks[h] * 1.4426950408889634f;
            const float top = fmaxf(c[h].m, sink);
            const float shrink = exp2f(c[h].m - top);
            inv = shrink / (l * shrink + exp2f(sink - top));
        }
#pragma unroll
        for (int t = 0; t < HD / 16; ++t) {
            if (t * 16 >= v_dim) break;
            u32x2 packed = {pack_bf16(c[h].o[t][0] * inv, c[h].o[t][1] * inv), pack_bf16(c[h].o[t][2] * inv, c[h].o[t][3] * inv)};
            *reinterpret_cast<u32x2*>(dest + (size_t)h * v_dim + t * 16 + g * 4) = packed;
        }
    }
}

template <int HD>
__device__ __forceinline__ void load_query(Columns<HD>& c, const uint16_t* __restrict__ q_row, int head_dim, bool valid) {
    const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int dc = 0; dc < HD / 32; ++dc) {
        c.q[dc] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
        if (valid && dc * 32 + g * 8 < head_dim) c.q[dc] = *reinterpret_cast<const bf16x8*>(q_row + dc * 32 + g * 8);
    }
#pragma unroll
    for (int t = 0; t < HD / 16; ++t) c.o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    c.m = NEG_BIG;
    c.l = 0.0f;
}

// ---- prompt portions ---------------------------------------------------------------------------
// A workgroup per (tile of 64 query rows, kv head, run of NH query heads of its group), numbered
// tile by tile in the order the caller lists the tiles (those that see the most keys first: the
// short ones then fill in behind, whatever head they belong to); four waves, 16
// rows each, every wave with the same NH heads: a page's keys and values are read once for all
// of them (from global memory and from LDS), which is what a long context is bound by. Fewer
// heads per workgroup give more and shorter workgroups, which evens out a short causal prompt.
// The pages of
// the kv head are copied global -> registers (two pages ahead) -> LDS (one page ahead of the
// one being worked on; two LDS buffers, one barrier per page), so that the copy hides behind the
// softmax arithmetic. tile_seg / tile_row0: the segment of each tile and its first row (a tile never
// spans two segments). LDS rows are padded by 16 bytes against bank conflicts.
#define KV_PAD 8
// Where the kernel needs no more than 256 registers a wave it says so (two waves per SIMD at
// least): the compiler then keeps the MFMA results in ordinary registers. Left with all 512 it puts
// them into the accumulation registers, and the softmax's rescaling of the output and the masks on
// the scores then cost a move out and a move back per value and page (112 + 80 of the ~560 vector
// instructions of two pages).
//
// PARTS 2: eight waves, the pages shared out between two halves of four waves (every second page each, with buffers
// of its own), which merge at the end, the first half's rows first. With NH 2 every key and value read from LDS serves
// two heads, and there are as many waves as with one half and NH 1. (The reads from LDS, 16 KB a wave and page, bound the
// kernel beside the softmax: one head 452 TFLOP/s over a prompt of 32,768 tokens, 16 heads in 8 groups; two heads in halves
// 560.)
template <int HD, int NH, int PARTS>
__global__ __launch_bounds__(256 * PARTS) __attribute__((amdgpu_waves_per_eu((HD <= 64 && NH <= 2) ? 2 : 1))) void attention_prefill_kernel(
    const uint16_t* __restrict__ q, uint16_t* __restrict__ out, const uint16_t* __restrict__ k_pages,
    const uint16_t* __restrict__ v_pages, const int32_t* __restrict__ block_table, int table_stride,
    const int32_t* __restrict__ tile_seg, const int32_t* __restrict__ tile_row0, const int32_t* __restrict__ seg_row0,
    const int32_t* __restrict__ row_pos, int num_heads, int num_kv_heads, int head_dim, int v_dim, float scale_log2, int window,
    int chunk, float cap, float cap_scale, int keep_first, const float* __restrict__ sinks, const float* __restrict__ slopes) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    // a key's row in LDS holds HD channels, those past head_dim zero: every lane loads its operand
    constexpr int k_stride = HD + KV_PAD;
    const int v_stride = PAGE + KV_PAD;
    const int k_elems = PAGE * k_stride, v_elems = v_dim * v_stride;
    const int half = PARTS > 1 ? threadIdx.x >> 8 : 0, tid = threadIdx.x & 255;
    uint16_t* lds = reinterpret_cast<uint16_t*>(lds_raw) + (size_t)half * 2 * (k_elems + v_elems);     // [half][buffer][K tile | V tile]
    if (head_dim < HD) {
        const int runs_per_row = (HD - head_dim) / 8;          // head_dim is a multiple of 16
        for (int run = tid; run < 2 * PAGE * runs_per_row; run += 256) {
            const int buffer = run / (PAGE * runs_per_row), row = run / runs_per_row % PAGE, at = run % runs_per_row;
            *reinterpret_cast<u32x4*>(lds + (size_t)buffer * (k_elems + v_elems) + row * k_stride + head_dim + at * 8) = u32x4{0u, 0u, 0u, 0u};
        }
    }

    const int group = num_heads / num_kv_heads, runs = (group + NH - 1) / NH;
    const int per_tile = num_kv_heads * runs;
    const int tile = blockIdx.x / per_tile, of_tile = blockIdx.x % per_tile;
    const int kvh = of_tile / runs, first_in_group = (of_tile % runs) * NH;
    const int lane = tid & 63, wave = tid >> 6, col = lane & 15, g = lane >> 4;
    const int seg = tile_seg[tile];
    const int tile_first_row = tile_row0[tile];
    const int seg_end = seg_row0[seg + 1];
    const int tile_rows = seg_end - tile_first_row < 64 ? seg_end - tile_first_row : 64;
    const int row0 = tile_first_row + wave * 16;                        // this wave's rows
    const int rows = tile_rows - wave * 16 < 16 ? tile_rows - wave * 16 : 16;     // may be <= 0
    const bool valid = col < rows;
    const int my_row = valid ? row0 + col : tile_first_row;
    const int my_pos = row_pos[my_row];
    const int wave_hi = rows > 0 ? row_pos[row0 + rows - 1] : -1;       // last position of this wave
    const int pos_lo = row_pos[tile_first_row], pos_hi = row_pos[tile_first_row + tile_rows - 1];
    const int my_first = fw_first_visible(my_pos, window, chunk);
    const int tile_first = fw_first_visible(pos_lo, window, chunk);      // the first key never falls as the position rises

    // a head past the end of the group computes along on zeros and is not stored
    Columns<HD> c[NH];
#pragma unroll
    for (int h = 0; h < NH; ++h) {
        const bool head_there = first_in_group + h < group;
        const int head = kvh * group + (head_there ? first_in_group + h : 0);
        load_query<HD>(c[h], q + ((size_t)my_row * num_heads + head) * head_dim, head_dim, valid && head_there);
    }
    const int32_t* table = block_table + (size_t)seg * table_stride;
    const size_t k_page_elems = (size_t)PAGE * head_dim, v_page_elems = (size_t)PAGE * v_dim;

    // the copy: a page's K is 64 rows of head_dim, its V v_dim rows of 64; runs of 16 bytes.
    // Loads are unconditional (a run or a page past the end is read from a valid place again and
    // never used) and the barriers order LDS traffic only, so that the pages requested stay in
    // flight while the page before them is worked on.
    const int k_runs = PAGE * head_dim / 8, v_runs = PAGE * v_dim / 8;
    constexpr int MAX_RUNS = HD * PAGE / 8 / 256;                                // per thread, per operand
    // The pages a tile walks: those of the kept first keys that lie before the window's first page, then
    // the window's. `step` numbers them; block_of gives the page's place in the sequence.
    const int window_block = tile_first / PAGE, last_block = pos_hi / PAGE;
    const int kept_blocks = (keep_first + PAGE - 1) / PAGE < window_block ? (keep_first + PAGE - 1) / PAGE : window_block;
    const int last_step = kept_blocks + last_block - window_block;
    auto block_of = [&](int step) { return step < kept_blocks ? step : window_block + step - kept_blocks; };
    u32x4 hold_k0[MAX_RUNS], hold_v0[MAX_RUNS], hold_k1[MAX_RUNS], hold_v1[MAX_RUNS];
    // what a thread copies of every page: fixed offsets, so that a page's address is a scalar
    // base plus these (no vector arithmetic per page; the registers that receive a page are
    // otherwise borrowed for it, and giving them back means waiting for loads still in flight)
    uint32_t run_offset[MAX_RUNS], run_offset_v[MAX_RUNS];
#pragma unroll
    for (int u = 0; u < MAX_RUNS; ++u) {
        run_offset[u] = (uint32_t)(tid + u * 256 < k_runs ? tid + u * 256 : 0) * 8u;
        run_offset_v[u] = (uint32_t)(tid + u * 256 < v_runs ? tid + u * 256 : 0) * 8u;
    }
    auto fetch = [&](u32x4 (&hold_k)[MAX_RUNS], u32x4 (&hold_v)[MAX_RUNS], int step) {
        const int page = __builtin_amdgcn_readfirstlane(table[block_of(step < last_step ? step : last_step)]);
        const uint16_t* k_from = k_pages + ((size_t)page * num_kv_heads + kvh) * k_page_elems;
        const uint16_t* v_from = v_pages + ((size_t)page * num_kv_heads + kvh) * v_page_elems;
#pragma unroll
        for (int u = 0; u < MAX_RUNS; ++u) {
            hold_k[u] = *reinterpret_cast<const u32x4*>(k_from + run_offset[u]);
            hold_v[u] = *reinterpret_cast<const u32x4*>(v_from + run_offset_v[u]);
        }
    };
    // The values of keys past the last one written (only in the tile's last page) are zeroed on
    // their way to LDS: whatever an earlier owner of the page left there must not meet P = 0.
    auto stash = [&](const u32x4 (&hold_k)[MAX_RUNS], const u32x4 (&hold_v)[MAX_RUNS], int buffer, int step) {
        const int block = block_of(step);
        uint16_t* kt = lds + (size_t)buffer * (k_elems + v_elems);
        uint16_t* vt = kt + k_elems;
        const int k_per_row = head_dim / 8;
        const int last_written = pos_hi - block * PAGE;         // < 0 for a page past the end: never attended
#pragma unroll
        for (int u = 0; u < MAX_RUNS; ++u) {
            const int run = tid + u * 256;
            if (run < k_runs) *reinterpret_cast<u32x4*>(kt + (run / k_per_row) * k_stride + (run % k_per_row) * 8) = hold_k[u];
            if (run < v_runs) {
                u32x4 v = hold_v[u];
                if (last_written < PAGE - 1) {
                    const int key0 = (run % 8) * 8;             // this run: keys key0 .. key0 + 7 of one channel
#pragma unroll
                    for (int word = 0; word < 4; ++word) {
                        const int first_key = key0 + 2 * word;
                        v[word] &= first_key + 1 <= last_written ? 0xffffffffu : (first_key <= last_written ? 0xffffu : 0u);
                    }
                }
                *reinterpret_cast<u32x4*>(vt + (run / 8) * v_stride + (run % 8) * 8) = v;
            }
        }
    };
    // the heads' slopes of a bias by distance, in the units of the raw scores (which scale_log2 turns into the exponent's)
    float dist[NH];
#pragma unroll
    for (int h = 0; h < NH; ++h)
        dist[h] = (slopes && first_in_group + h < group) ? slopes[kvh * group + first_in_group + h] * 1.4426950408889634f / scale_log2 : 0.0f;
    auto attend = [&](int step, int buffer) {
        const int base = block_of(step) * PAGE;
        if (rows > 0 && base <= wave_hi) {      // a wave whose rows all lie before this page has nothing to add
            const uint16_t* kt = lds + (size_t)buffer * (k_elems + v_elems);
            // a lane without a row computes along with the bounds of the tile's first row (nothing of
            // it is stored): a page that is whole for the rows is then whole for the wave
            attend_page<HD, NH, false, true>(c, kt, kt + k_elems, head_dim, v_dim, scale_log2, my_first - base, my_pos - base, pos_hi - base,
                            k_stride, v_stride, cap, cap_scale, keep_first - base, slopes ? dist : nullptr);
        }
    };

    // a half's page number i travels: global -> register set i % 2, requested two pages ahead -> LDS
    // buffer i % 2, stored while page i - 1 is worked on -> attended
    auto step_of = [&](int i) { return PARTS * i + half; };
    const int pages = (last_step + PARTS) / PARTS;              // of the first half; the other may have one less (a page past the end)
    fetch(hold_k0, hold_v0, step_of(0));
    fetch(hold_k1, hold_v1, step_of(1));
    stash(hold_k0, hold_v0, 0, step_of(0));
    fw_lds_barrier();
    for (int i = 0; i < pages; i += 2) {
        fetch(hold_k0, hold_v0, step_of(i + 2));
        __builtin_amdgcn_sched_barrier(0);      // keep the requests ahead of the work they overlap
        attend(step_of(i), 0);
        stash(hold_k1, hold_v1, 1, step_of(i + 1));
        fw_lds_barrier();
        if (i + 1 >= pages) break;
        fetch(hold_k1, hold_v1, step_of(i + 3));
        __builtin_amdgcn_sched_barrier(0);
        attend(step_of(i + 1), 1);
        stash(hold_k0, hold_v0, 0, step_of(i + 2));
        fw_lds_barrier();
    }
    if constexpr (PARTS > 1) {
        float* left = reinterpret_cast<float*>(lds_raw) + tid;
        __syncthreads();
        if (half == 1) leave_columns(c, left);
        __syncthreads();
        if (half == 1) return;
        join_columns(c, left);
    }
    const int first_head = kvh * group + first_in_group;
    store_columns(c, valid, group - first_in_group, sinks ? sinks + first_head : nullptr, out + ((size_t)my_row * num_heads + first_head) * v_dim, v_dim);
}

// ---- prompt portions, heads of 64 or 128 channels two by two ------------------------------------
// The same tiles and workgroups' order; a wave has 16 rows of two query heads of a kv group, so that an operand read from LDS serves
// both. What it is bound by is the softmax: 168 vector instructions a wave and page, 34 of them exponentials at half the rate, about twice the clocks of
// its 32 products (HD 64). So a wave's loop holds three pages at once: while the softmax of page i runs, the
// matrix pipe works on the scores of page i + 1 and on the output of page i - 1, a product or two behind every few vector instructions, a
// load behind every few more (issued together behind the barrier, eight waves' loads keep a compute unit's memory path for as long as a third of a page).
// us, one head a workgroup or halves of attend_page / this: 16 heads in 8 groups of 64 channels, 2,048 rows behind 30,720 keys 442 / 359 (741 TFLOP/s), 32
// heads behind 2,048 98 / 80, 6,144 rows behind 8,192 956 / 690 (822); 16 heads in 4 groups of 128, 2,048 rows with a window of 1,024 44.7 / 29.0, behind
// 4,096 187 / 104 (828). In halves the eight waves meet at one barrier a page, which costs a tenth of what four-wave workgroups side by side reach. Three waves a
// SIMD (168 registers) gave 3 % with work for all of them and spilled.
//
//  * keys and values travel straight into LDS (buffer_load .. lds), STG stages of each; rows are not padded, their 16-byte chunks are
//    stored permuted so that a wave's reads meet no bank twice;
//  * the 16 keys of a score tile are chosen so that a lane's eight scores of two tiles are those of eight keys in a row: key
//    32 (tile / 2) + 8 (row / 4) + 4 (tile % 2) + row % 4. The second product's operand is then one 16-byte read of a channel's keys;
//  * values past the last one written (a tile's last page) are zeroed in LDS ahead of their product.
//
// PARTS 2: eight waves, the pages dealt to two halves of four waves with stages of their own, which merge at the end.
// The largest of three scores in one instruction. (fmaxf makes two, and one more for every score to quiet what might be a signalling NaN.) What
// a matrix product has written is read here only behind fw_mfma_drain: the compiler does not see into the assembly.
__device__ __forceinline__ float max_of(float a, float b, float c) {
    float m;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(m) : "v"(a), "v"(b), "v"(c));
    return m;
}
__device__ __forceinline__ float quad_max_of(float x) {
    float a, b, c, d;
    fw_quad_partners16(x, a, b);
    asm("v_max_f32 %0, %1, %2" : "=v"(c) : "v"(a), "v"(b));
    fw_quad_partners32(c, a, b);
    asm("v_max_f32 %0, %1, %2" : "=v"(d) : "v"(a), "v"(b));
    return d;
}

template <int HD, int PARTS, int STG>
__global__ __launch_bounds__(256 * PARTS) __attribute__((amdgpu_waves_per_eu(2, 2))) void attention_prompt_kernel(
    const uint16_t* __restrict__ q, uint16_t* __restrict__ out, const uint16_t* __restrict__ k_pages,
    const uint16_t* __restrict__ v_pages, const int32_t* __restrict__ block_table, int table_stride,
    const int32_t* __restrict__ tile_seg, const int32_t* __restrict__ tile_row0, const int32_t* __restrict__ seg_row0,
    const int32_t* __restrict__ row_pos, int num_heads, int num_kv_heads, float scale_log2, int window,
    int chunk, float cap, float cap_scale, int keep_first, const float* __restrict__ sinks, const float* __restrict__ slopes) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds_raw[];     // [half][K stages | V stages]
    constexpr int NH = 2, DC = HD / 32, VT = HD / 16;
    constexpr int TILE = PAGE * HD * 2, LOADS = TILE / 4096;             // bytes of a page's keys (values) of a kv head; wave-wide loads per wave
    constexpr int K_CHUNKS = HD / 8, K_ROWS = 64 / K_CHUNKS;            // chunks of a key's row, rows of a wave-wide load
    const int half = PARTS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0, tid = threadIdx.x & 255;
    unsigned char* lds = lds_raw + (size_t)half * 2 * STG * TILE;
    unsigned char* lds_v = lds + STG * TILE;

    const int group = num_heads / num_kv_heads, runs = group / NH;
    const int per_tile = num_kv_heads * runs;
    const int tile = blockIdx.x / per_tile, of_tile = blockIdx.x % per_tile;
    const int kvh = of_tile / runs, first_head = kvh * group + (of_tile % runs) * NH;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i16 = lane & 15, g = lane >> 4;
    const int seg = tile_seg[tile];
    const int tile_first_row = tile_row0[tile];
    const int seg_end = seg_row0[seg + 1];
    const int tile_rows = seg_end - tile_first_row < 64 ? seg_end - tile_first_row : 64;
    const int row0 = tile_first_row + wave * 16;
    const int rows = tile_rows - wave * 16 < 16 ? tile_rows - wave * 16 : 16;     // may be <= 0
    const bool valid = i16 < rows;
    const int my_row = valid ? row0 + i16 : tile_first_row;      // a lane without a row computes along with the tile's first and is not stored
    const int my_pos = row_pos[my_row];
    const int pos_lo = row_pos[tile_first_row], pos_hi = row_pos[tile_first_row + tile_rows - 1];
    const int my_first = fw_first_visible(my_pos, window, chunk);
    const int tile_first = fw_first_visible(pos_lo, window, chunk);

    // The pages a tile walks: those of the kept first keys that lie before the window's first page, then the window's.
    const int window_block = tile_first / PAGE, last_block = pos_hi / PAGE;
    const int kept_blocks = (keep_first + PAGE - 1) / PAGE < window_block ? (keep_first + PAGE - 1) / PAGE : window_block;
    const int last_step = kept_blocks + last_block - window_block;
    auto block_of = [&](int step) { return step < kept_blocks ? step : window_block + step - kept_blocks; };
    auto step_of = [&](int i) { return PARTS * i + half; };
    const int pages = (last_step + PARTS) / PARTS;              // of the first half; the other may have one less (a page past the end, masked whole)
    const int32_t* table = block_table + (size_t)seg * table_stride;

    // what this lane asks for of a page: the chunk whose slot it fills
    uint32_t k_at[LOADS], v_at[LOADS];
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
        const int key = (wave * LOADS + j) * K_ROWS + lane / K_CHUNKS;
        const int swap = HD == 64 ? ((key >> 1) & 1) | (((key >> 3) & 3) << 1) : (key & 3) | (((key >> 3) & 3) << 2);
        k_at[j] = key * (HD * 2) + ((lane % K_CHUNKS) ^ swap) * 16;
        const int channel = (wave * LOADS + j) * 8 + (lane >> 3);
        v_at[j] = channel * (PAGE * 2) + ((lane & 7) ^ ((channel >> 1) & 7)) * 16;
    }
    // The numbers of 64 pages at a time, one a lane, and those of the next 64 on their way: a page's number read when it is needed would
    // stand between a barrier and the loads behind it. (Past the end: the last one again, never counted.)
    auto numbers = [&](int first) {
        const int step = step_of(first + lane);
        return table[block_of(step < last_step ? step : last_step)];
    };
    int held = numbers(0), ahead = numbers(64);
    int page_k = 0, page_before = 0, page_v = 0;                // of keys i, i - 1, i - 2; values follow the keys by two
    auto next_page = [&](int i) {
        page_v = page_before;
        page_before = page_k;
        page_k = __builtin_amdgcn_readlane(held, i & 63);
        if ((i & 63) == 63) {
            held = ahead;
            ahead = numbers(i + 65);
        }
    };
    // load number `u` of a page: LOADS of keys i, then as many of values i - 2
    auto request = [&](int i, int u) {
        if (u < LOADS) {
            const fw_buffer keys = fw_make_buffer(k_pages + ((size_t)page_k * num_kv_heads + kvh) * (PAGE * HD));
            fw_buffer_to_lds(keys, lds + (i % STG) * TILE + (wave * LOADS + u) * 1024, k_at[u], 0);
        } else {
            const fw_buffer channels = fw_make_buffer(v_pages + ((size_t)page_v * num_kv_heads + kvh) * (PAGE * HD));
            fw_buffer_to_lds(channels, lds_v + ((i + STG - 2) % STG) * TILE + (wave * LOADS + u - LOADS) * 1024, v_at[u - LOADS], 0);
        }
    };

    Columns<HD> c[NH];
#pragma unroll
    for (int h = 0; h < NH; ++h) load_query<HD>(c[h], q + ((size_t)my_row * num_heads + first_head + h) * HD, HD, valid);
    float dist[NH];
#pragma unroll
    for (int h = 0; h < NH; ++h) dist[h] = slopes ? slopes[first_head + h] * 1.4426950408889634f / scale_log2 : 0.0f;

    // operands: unit u < PV_UNITS is a run of 32 keys of 16 channels of the values, the others 32 channels of 16 keys
    constexpr int PV_UNITS = 2 * VT, UNITS = PV_UNITS + 4 * DC;
    const int k_swap = HD == 64 ? ((i16 >> 1) & 1) | ((i16 >> 2) << 1) : i16;
    const int k_row = (8 * (i16 >> 2) + (i16 & 3)) * (HD * 2);
    int k_lane[DC], v_lane[2];
#pragma unroll
    for (int d = 0; d < DC; ++d) k_lane[d] = k_row + ((d * 4 + g) ^ k_swap) * 16;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) v_lane[kb] = i16 * (PAGE * 2) + ((kb * 4 + g) ^ ((i16 >> 1) & 7)) * 16;
    auto read_k = [&](const unsigned char* stage, int kt, int d) {
        return *reinterpret_cast<const bf16x8*>(stage + k_lane[d] + (32 * (kt >> 1) + 4 * (kt & 1)) * (HD * 2));
    };
    auto read_v = [&](const unsigned char* stage, int kb, int t) { return *reinterpret_cast<const bf16x8*>(stage + v_lane[kb] + t * 16 * (PAGE * 2)); };
    // (two tiles of keys in turn, so that a product does not wait for the one it adds to)
    auto tile_of = [](int u) { return 2 * ((u - PV_UNITS) / (2 * DC)) + (u - PV_UNITS) % 2; };
    auto run_of = [](int u) { return (u - PV_UNITS) / 2 % DC; };
    auto operand = [&](const unsigned char* k_stage, const unsigned char* v_stage, int u) {
        return u < PV_UNITS ? read_v(v_stage, u / VT, u % VT) : read_k(k_stage, tile_of(u), run_of(u));
    };

    f32x4 s0[NH][4], s1[NH][4];
    uint32_t p0[NH][4][2], p1[NH][4][2];
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    auto work = [&](int u, const bf16x8& x, const uint32_t (&p)[NH][4][2], f32x4 (&s)[NH][4]) {
#pragma unroll
        for (int h = 0; h < NH; ++h) {
            if (u < PV_UNITS) {
                const int kb = u / VT, t = u % VT;
                const u32x4 pw = {p[h][2 * kb][0], p[h][2 * kb][1], p[h][2 * kb + 1][0], p[h][2 * kb + 1][1]};
                c[h].o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, __builtin_bit_cast(bf16x8, pw), c[h].o[t], 0, 0, 0);
            } else {
                const int kt = tile_of(u), d = run_of(u);
                s[h][kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, c[h].q[d], d ? s[h][kt] : zero, 0, 0, 0);
            }
        }
    };
    auto landed = [&](bool first) {
        if (first) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((2 * STG - 3) * LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STG - 2) * 2 * LOADS) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    // One page: the softmax of scores `s` into `p`, beside it the output of the page before (weights `p_before`) and the scores of the next.
    auto page = [&](int i, f32x4 (&s)[NH][4], f32x4 (&s_next)[NH][4], uint32_t (&p)[NH][4][2], const uint32_t (&p_before)[NH][4][2]) {
        landed(false);
        next_page(i + STG);
        const int base = block_of(step_of(i)) * PAGE;           // (past the end: beyond every position)
        const int lo = my_first - base, hi = my_pos - base, kept = keep_first - base;
        if (cap > 0.0f) {       // s <- cap * tanh(s * scale / cap), as attend_page
            const float twice = 2.0f * cap_scale * 1.4426950408889634f;
#pragma unroll
            for (int h = 0; h < NH; ++h)
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float e = __builtin_amdgcn_exp2f(s[h][kt][r] * twice);
                        s[h][kt][r] = cap - 2.0f * cap * __builtin_amdgcn_rcpf(1.0f + e);
                    }
        }
        if (slopes) {
#pragma unroll
            for (int h = 0; h < NH; ++h)
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        s[h][kt][r] = fmaf(-dist[h], (float)(hi - (32 * (kt >> 1) + 8 * g + 4 * (kt & 1) + r)), s[h][kt][r]);
        }
        if (!__all((lo <= 0 || kept >= lo) && hi >= PAGE - 1)) {
#pragma unroll
            for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int key = 32 * (kt >> 1) + 8 * g + 4 * (kt & 1) + r;
                    const bool seen = (key >= lo || key < kept) && key <= hi;
#pragma unroll
                    for (int h = 0; h < NH; ++h) s[h][kt][r] = seen ? s[h][kt][r] : NEG_BIG;
                }
        }
        const unsigned char* k_stage = lds + ((i + 1) % STG) * TILE;
        const unsigned char* v_stage = lds_v + ((i + STG - 1) % STG) * TILE;
        // SLOTS runs of vector instructions, the units of products dealt to them evenly, an operand read AHEAD units before its product
        constexpr int SLOTS = 14, AHEAD = HD == 64 ? 6 : 2;
        bf16x8 ring[AHEAD + 1];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) ring[u] = operand(k_stage, v_stage, u);
        auto units = [&](int slot) {
#pragma unroll
            for (int u = 0; u < 2 * LOADS; ++u)         // (a compute unit takes a wave's load in 16 clocks: all at once, they would be waited for)
                if (u * SLOTS / (2 * LOADS) == slot) request(i + STG, u);
#pragma unroll
            for (int u = 0; u < UNITS; ++u)
                if (u * SLOTS / UNITS == slot) {
                    if (u + AHEAD < UNITS) ring[(u + AHEAD) % (AHEAD + 1)] = operand(k_stage, v_stage, u + AHEAD);
                    work(u, ring[u % (AHEAD + 1)], p_before, s_next);
                }
        };
        float top[NH], alpha[NH], shift[NH], sum[NH];
        bool rose = false;
#pragma unroll
        for (int h = 0; h < NH; ++h) {
#pragma unroll
            for (int part = 0; part < 2; ++part) {
                units(h * 3 + part);
                const f32x4 &a = s[h][2 * part], &b = s[h][2 * part + 1];
                top[h] = max_of(part ? top[h] : a[0], a[0], a[1]);
                top[h] = max_of(top[h], a[2], a[3]);
                top[h] = max_of(top[h], b[0], b[1]);
                top[h] = max_of(top[h], b[2], b[3]);
                __builtin_amdgcn_sched_barrier(0);
            }
            units(h * 3 + 2);
            const float page_max = quad_max_of(top[h]);
            // a column that has seen no key yet keeps NEG_BIG (the raw maximum times the scale would overflow)
            const float new_max = fmaxf(c[h].m, page_max > 0.5f * NEG_BIG ? page_max * scale_log2 : NEG_BIG);
            alpha[h] = __builtin_amdgcn_exp2f(c[h].m - new_max);
            rose |= alpha[h] != 1.0f;
            c[h].m = new_max;
            shift[h] = new_max > 0.5f * NEG_BIG ? -new_max : 0.0f;
            sum[h] = 0.0f;
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
                units(6 + h * 4 + kt);
                float e[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) e[r] = __builtin_amdgcn_exp2f(fmaf(s[h][kt][r], scale_log2, shift[h]));
                sum[h] += (e[0] + e[1]) + (e[2] + e[3]);
                p[h][kt][0] = pack_bf16_pair(e[0], e[1]);
                p[h][kt][1] = pack_bf16_pair(e[2], e[3]);
                asm volatile("" : "+v"(p[h][kt][0]), "+v"(p[h][kt][1]), "+v"(sum[h]));      // here, among the products, and not behind the branch below
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
        for (int h = 0; h < NH; ++h) c[h].l = c[h].l * alpha[h] + sum[h];
        fw_mfma_drain();            // a branch follows that leads to code reading what the products wrote
        if (__any(rose)) {          // the output holds the pages up to i - 1 now
#pragma unroll
            for (int h = 0; h < NH; ++h)
#pragma unroll
                for (int t = 0; t < VT; ++t) c[h].o[t] *= alpha[h];
        }
    };

    // the stage of the values of "page -1", whose weights are zero
#pragma unroll
    for (int u = 0; u < TILE / 4096; ++u) *reinterpret_cast<u32x4*>(lds_v + (STG - 1) * TILE + (u * 256 + tid) * 16) = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) p1[h][kt][0] = p1[h][kt][1] = 0u;
#pragma unroll
    for (int i = 0; i < STG; ++i) {
        next_page(i);
#pragma unroll
        for (int u = 0; u < (i < 2 ? LOADS : 2 * LOADS); ++u) request(i, u);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    landed(true);
    {
        const unsigned char* k_stage = lds;
#pragma unroll
        for (int u = PV_UNITS; u < UNITS; ++u) work(u, operand(k_stage, lds_v, u), p1, s0);
        fw_mfma_drain();
    }
    int i = 0;
    for (; i + 1 < pages; i += 2) {
        page(i, s0, s1, p0, p1);
        page(i + 1, s1, s0, p1, p0);
    }
    if (i < pages) page(i, s0, s1, p0, p1);
    // the output of the last page: the values past the last one written are zeroed first (whatever an earlier owner of the page left there
    // must not meet a weight of 0)
    const int last = pages - 1;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    unsigned char* v_last = lds_v + (last % STG) * TILE;
    const int last_written = step_of(last) >= last_step ? pos_hi - last_block * PAGE : PAGE - 1;
    if (last_written < PAGE - 1) {
        for (int run = tid; run < HD * 8; run += 256) {
            const int channel = run >> 3, first_key = ((run & 7) ^ ((channel >> 1) & 7)) * 8;
            u32x4* at = reinterpret_cast<u32x4*>(v_last + run * 16);
            u32x4 v = *at;
#pragma unroll
            for (int word = 0; word < 4; ++word) {
                const int key = first_key + 2 * word;
                v[word] &= key + 1 <= last_written ? 0xffffffffu : (key <= last_written ? 0xffffu : 0u);
            }
            *at = v;
        }
    }
    __syncthreads();
    if (pages & 1) {
#pragma unroll
        for (int u = 0; u < PV_UNITS; ++u) work(u, operand(lds, v_last, u), p0, s1);
    } else {
#pragma unroll
        for (int u = 0; u < PV_UNITS; ++u) work(u, operand(lds, v_last, u), p1, s0);
    }
    fw_mfma_drain();
    if constexpr (PARTS > 1) {
        float* left = reinterpret_cast<float*>(lds_raw) + tid;
        __syncthreads();
        if (half == 1) leave_columns(c, left);
        __syncthreads();
        if (half == 1) return;
        join_columns(c, left);
    }
    store_columns(c, valid, NH, sinks ? sinks + first_head : nullptr, out + ((size_t)my_row * num_heads + first_head) * HD, HD);
}

// ---- decode ------------------------------------------------------------------------------------
#define MERGE_PARTS 64               // parts of a row up to which the last workgroup keeps their weights in LDS (a context of 16,384 tokens at one run each)
// How a step is cut into workgroups. Where the rows are equally long, into whole splits of every row that fill the compute units once, each with a workgroup
// of its own, so that all end together; where that leaves more than three tenths of them idle and the rows have LONG_RUNS runs, twice or three
// times. Counted are the places of the grid, those of rows that fill a recorded step up among them: a workgroup that ends at once has still moved
// the next one on by a compute unit. us of the best of 1 to 24 splits / this rule / as many splits as bring all the rows' runs below 256, mean of 560
// steps (1 to 96 rows, a third of them filled up, 300 to 6,000 keys; 1 to 8 kv heads of 64 and 128 channels) 1 / 1.021 / 1.057: 20 rows filled up to 24 behind
// 2,900 keys, 32 heads in 8 groups of 64 channels 28.0 / 28.0 / 33.3, 2 groups of 16 heads of 128 channels 24.6 / 24.6 / 32.0; 24 rows, 4 groups of 128
// channels 37.6 / 37.6 / 47.0; 40 rows, the same, 1,000 keys (1 and 2 splits) 24.3 and 30.9, 2,900 (1, 2 and 3) 58.3, 65.4 and 51.7. Heads of 144 to
// 256 channels, which do not stream, are cut the same way: 230 steps, the best 1, by this rule 1.015, 1.028 with 256 workgroups (384 where rows fill the step up); 48
// rows of 1,000 keys, 4 groups of 256 channels 55.5 by this rule, 63.1 by those, but of 2,900 keys 135.6 and 122.5.
// Where the lengths differ, RAGGED_WORKGROUPS at most (rounds rounded up): a half more than compute units fill up behind those of short rows. Mean of 48
// ragged steps (3 to 64 rows of up to 6,000 keys, 4 head shapes of 64 and 128 channels) with 256 / 320 / 384 / 512 workgroups 41.4 / 40.5 / 39.7 / 40.1 us.
#define EVEN_WORKGROUPS 256
#define RAGGED_WORKGROUPS 384
#define LONG_RUNS 8
struct EvenSplits {
    int plain, many;        // of a row; from LONG_RUNS runs on
    int runs;               // that a window leaves of a row, most of the time (a row whose window ends inside a page sees a page more)
};
static EvenSplits even_splits(int rows, int across, int max_splits, int span, int keep_first) {
    const int places = rows > 3 * EVEN_WORKGROUPS ? rows : rows * across;       // of one split
    EvenSplits even = {places < EVEN_WORKGROUPS ? EVEN_WORKGROUPS / places : 1, 0, max_splits};
    for (int times = 1; times <= 3 && even.many == 0; ++times) {
        const int splits = times * EVEN_WORKGROUPS / places;
        if (10 * splits * places >= 7 * times * EVEN_WORKGROUPS) even.many = splits;
    }
    if (even.many == 0) even.many = places < 3 * EVEN_WORKGROUPS ? 3 * EVEN_WORKGROUPS / places : 1;
    if (span > 0) {
        const int pages = (span - 1) / PAGE + 1 + (keep_first + PAGE - 1) / PAGE, runs = (pages + SPLIT_PAGES - 1) / SPLIT_PAGES;
        even.runs = runs < max_splits ? runs : max_splits;
    }
    return even;
}
// grid (kv heads * head tiles, rows, splits), or the first two changed over beyond 65,535 rows; four waves, each takes one page of the split's
// SPLIT_PAGES, and their results are merged in LDS in the order of the keys. Columns are the
// query heads of the kv group (16 per head tile). partial [rows][heads][max_splits][v_dim + 4]:
// unnormalised output, then maximum and sum; a split with nothing to do writes nothing and takes
// no ticket. The last workgroup of a (row, kv head, head tile) to arrive merges what the others
// left; the only workgroup of a short row writes the result at once.
// What bounds it is memory: bytes on their way to the compute units, for as long as the walk takes. Up to 128 channels a wave's
// loads of a page's keys go out as soon as the page before has been scored, those of its values as soon as the values before are used, the
// page's number one page earlier still, and the first page's while the fused variant forms the queries; each page in turn, with
// its number looked up in front and nothing on its way during the arithmetic (and cut into up to 512 workgroups): 64 rows of 725..2,900 keys, 32 heads in 8
// groups of 64 channels 72.6 us, now 54.8 (4.6 TB/s); 24 rows 35.3, now 30.5; 8 rows of 2,048 keys 15.7, now 14.6; 8 rows of 32,768 keys, 16 heads
// 101.5, now 100.4 (5.4 TB/s); 16 heads in one group of 128 channels, 64 rows 40.1, now 33.1. Two pages in the registers at a time did not fit (the compiler
// copies between them and spills); 167 registers leave room for three waves a SIMD.
// What the fused variant does in front of the attention: the step's raw projections (float32
// [rows][(heads + kv heads) * head_dim + kv heads * v_dim]: queries, keys, values) get their per-head RMS norm and
// rotation here, as qk_norm_rope_kv_write does in a kernel of its own (the same arithmetic in the
// same order), so that a decode step needs no such kernel. Every workgroup norms and rotates the
// query heads it works on; the workgroup whose pages include the row's own position also norms and
// rotates the new key, stores it and the new value in their page, and reads them back from there
// with the rest of the page (its own stores, ordered by a workgroup barrier).
struct FusedProjections {
    const float* qkv;               // null: q holds finished bfloat16 queries and the cache is up to date
    const float* q_norm_weight;     // [head_dim] or null
    const float* k_norm_weight;
    float eps;
    const float* cos_table;         // [rows][rotary_dim / 2]
    const float* sin_table;
    int rotary_dim;
    int write_kv;                   // 0: another execution of the layer has stored this step's keys and values already
    int interleaved;                // 0: channel i turns with channel i + rotary_dim / 2; 1: channel 2i with channel 2i + 1
    int width;                      // floats of a row of qkv: queries alone where the keys and values are another layer's
    const float* q_row_scale;       // [rows] or null: a factor on the row's finished queries
};

// One head-vector of head_dim channels by one wave: optional RMS norm, then the half-split rotation
// of the first rotary_dim channels; `store(d, value)` takes the results. scratch: head_dim floats of
// LDS of the wave's own. (native/include/flyweight_v2_native_kernels.hpp:1015-1050)
template <typename Store>
__device__ __forceinline__ void norm_rotate_vector(const float* __restrict__ source, const float* __restrict__ weight, float eps,
                                                   const float* __restrict__ cos_row, const float* __restrict__ sin_row,
                                                   int rotary_dim, int head_dim, float* scratch, Store store, int interleaved = 0) {
    const int lane = threadIdx.x & 63;
    float inv = 1.0f;
    if (weight) {
        float sum = 0.0f;
        for (int d = lane; d < head_dim; d += 64) {
            const float v = source[d];
            sum += v * v;
        }
        sum = wave_sum(sum);
        inv = rsqrtf(sum / (float)head_dim + eps);
    }
    for (int d = lane; d < head_dim; d += 64) {
        const float v = source[d];
        scratch[d] = weight ? v * inv * weight[d] : v;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int half = rotary_dim / 2;
    for (int d = lane; d < head_dim; d += 64) {
        float value = scratch[d];
        if (d < rotary_dim) {
            const bool is_first = interleaved ? (d & 1) == 0 : d < half;
            const int pair = interleaved ? d >> 1 : (d < half ? d : d - half);
            const float other = scratch[interleaved ? d ^ 1 : (d < half ? d + half : d - half)];
            const float c = cos_row[pair], s = sin_row[pair];
            value = fmaf(value, c, is_first ? -(other * s) : other * s);
        }
        store(d, value);
    }
}

template <int HD, bool FUSED>
__global__ __launch_bounds__(64 * SPLIT_PAGES) __attribute__((amdgpu_waves_per_eu(HD <= 128 ? 2 : 1))) void attention_decode_split_kernel(
    const uint16_t* __restrict__ q, uint16_t* __restrict__ out, float* partial, int* tickets,
    uint16_t* k_pages, uint16_t* v_pages, const int32_t* __restrict__ block_table, int table_stride,
    const int32_t* __restrict__ row_seg, const int32_t* __restrict__ row_pos, int num_heads, int num_kv_heads,
    int head_dim, int v_dim, float scale_log2, int window, int chunk, float cap, float cap_scale, int max_splits,
    const int32_t* __restrict__ decode_work, const FusedProjections fused, int keep_first, const float* __restrict__ sinks,
    const float* __restrict__ slopes, bool heads_first, const EvenSplits even) {
    __shared__ f32x4 shared_o[SPLIT_PAGES][HD / 16][64];
    __shared__ float shared_m[SPLIT_PAGES][16], shared_l[SPLIT_PAGES][16];
    __shared__ int ticket_shared;
    __shared__ float merge_w[MERGE_PARTS][16], merge_l[MERGE_PARTS][16];
    __shared__ __attribute__((aligned(16))) uint16_t fused_q[FUSED ? 16 : 1][FUSED ? HD : 8];
    __shared__ float fused_scratch[FUSED ? SPLIT_PAGES : 1][FUSED ? HD : 1];
    const int row = heads_first ? blockIdx.y : blockIdx.x, across = heads_first ? blockIdx.x : blockIdx.y, split = blockIdx.z;
    const int rows = heads_first ? gridDim.y : gridDim.x, acrosses = heads_first ? gridDim.x : gridDim.y;
    const int group = num_heads / num_kv_heads;
    const int head_tiles = (group + 15) / 16;
    const int kvh = across / head_tiles, head_tile = across % head_tiles;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), col = lane & 15, g = lane >> 4;
    const int pos = row_pos[row];
    // asked for together with the position, not behind the branches below
    const int segment = row_seg[row], step_runs = *(decode_work ? decode_work : row_seg);
    const int first = fw_first_visible(pos, window, chunk);
    // The pages a row walks: those of the kept first keys that lie before the window's first page, then the
    // window's. They are numbered through (`step`), and the splits are counted over the steps.
    const int window_block = first / PAGE, last_block = pos / PAGE;
    const int kept_blocks = (keep_first + PAGE - 1) / PAGE < window_block ? (keep_first + PAGE - 1) / PAGE : window_block;
    const int last_step = kept_blocks + last_block - window_block;
    // Splits are counted from the first page that holds a visible key; a split is `rounds` runs of
    // SPLIT_PAGES pages, the same number for every row of the step. One run each serves while there are few; beyond, fewer and longer workgroups
    // read the cache faster, and a row has fewer parts to merge (one workgroup for a whole row needs no merge at all). decode_work says what
    // the step holds: below zero that its rows are equally long and the runs of the longest; else the runs of all rows together, of which no more
    // count than a window leaves of every row (rows that all reach it are equally long). Counting the step's work,
    // not the row's, gives a long row among short ones its share of the chip.
    int rounds = 1;
    if (decode_work) {
        if (step_runs < 0 || step_runs >= (long long)rows * even.runs) {
            const uint32_t seen = -(uint32_t)step_runs;
            const int longest = step_runs < 0 && seen < (uint32_t)even.runs ? (int)seen : even.runs;
            const int splits = longest >= LONG_RUNS ? even.many : even.plain;
            rounds = splits == 1 ? (int)gridDim.z : (longest + splits - 1) / splits;
        } else {
            rounds = (int)(((long long)step_runs * acrosses + RAGGED_WORKGROUPS - 1) / RAGGED_WORKGROUPS);
        }
        rounds = rounds < 1 ? 1 : rounds;
    }
    const int pages_per_split = SPLIT_PAGES * rounds;
    const int first_step = split * pages_per_split;
    if (first_step > last_step) return;         // the whole workgroup
    const int in_group = head_tile * 16 + col;
    const bool valid = in_group < group;
    const int head = kvh * group + (valid ? in_group : 0);

    Columns<HD> columns_of_wave[1];
    Columns<HD>& c = columns_of_wave[0];
    // the wave's pages: every SPLIT_PAGES-th step from its first one on; their numbers are asked for ahead
    const int my_first = first_step + wave;
    const int my_rounds = my_first > last_step ? 0 : (last_step - my_first) / SPLIT_PAGES + 1 < rounds ? (last_step - my_first) / SPLIT_PAGES + 1 : rounds;
    auto block_of = [&](int round) {
        const int step = my_first + round * SPLIT_PAGES;
        return step < kept_blocks ? step : window_block + step - kept_blocks;
    };
    const int32_t* table = block_table + (size_t)segment * table_stride;
    auto number_of = [&](int round) { return table[block_of(round < my_rounds ? round : my_rounds - 1)]; };
    // Up to 128 channels the pages stream: STAGES of them are on their way at any time, the first ones while the queries are formed.
    constexpr bool STREAMED = HD <= 128;
    constexpr int STAGES = 1;       // (written out without the loops over them the compiler keeps the pages otherwise: heads of 128 channels spill)
    PageOnWay<STREAMED ? HD : 32> pages[STAGES];
    const PageOffsets<STREAMED ? HD : 32> offsets(head_dim);
    int next[STAGES];
    auto keys_at = [&](int page, bool wanted) {
        return fw_make_buffer(k_pages + ((size_t)page * num_kv_heads + kvh) * PAGE * head_dim, wanted ? (uint32_t)(PAGE * head_dim * 2) : 0u);
    };
    auto values_at = [&](int page, bool wanted) {
        return fw_make_buffer(v_pages + ((size_t)page * num_kv_heads + kvh) * PAGE * v_dim, wanted ? (uint32_t)(PAGE * v_dim * 2) : 0u);
    };
    // this row's new key and value are stored below, and their page is asked for behind that
    const int own_round = FUSED && fused.write_kv && my_rounds > 0 && my_first + (my_rounds - 1) * SPLIT_PAGES == last_step ? my_rounds - 1 : -1;
    int first_page[STAGES];
    if (STREAMED && my_rounds > 0) {
#pragma unroll
        for (int i = 0; i < STAGES; ++i) {
            first_page[i] = number_of(i);
            next[i] = number_of(STAGES + i);
        }
#pragma unroll
        for (int i = 0; i < STAGES; ++i) {
            first_page[i] = __builtin_amdgcn_readfirstlane(first_page[i]);
            const bool wanted = i < my_rounds && i != own_round;
            ask_for_keys(pages[i], offsets, keys_at(first_page[i], wanted));
            ask_for_values(pages[i], offsets, values_at(first_page[i], wanted));
        }
    }
    if (FUSED) {
        const float* projections = fused.qkv + (size_t)row * fused.width;
        const int half = fused.rotary_dim / 2;
        const float* cos_row = fused.cos_table + (size_t)row * half;
        const float* sin_row = fused.sin_table + (size_t)row * half;
        const int columns = group - head_tile * 16 < 16 ? group - head_tile * 16 : 16;
        // the vectors of this workgroup: its query heads, then (where the row's own position lies
        // in its pages) the new key and the new value; a wave takes every fourth
        const bool stores = fused.write_kv && last_step < first_step + pages_per_split;
        const int vectors = columns + (stores ? 2 : 0);
        const int slot = pos % PAGE;
        const int own_page = stores ? block_table[(size_t)segment * table_stride + last_block] : 0;
        const float q_factor = fused.q_row_scale ? fused.q_row_scale[row] : 1.0f;
        for (int v = wave; v < vectors; v += SPLIT_PAGES) {
            if (v < columns) {
                uint16_t* dest = fused_q[v];
                norm_rotate_vector(projections + (size_t)(kvh * group + head_tile * 16 + v) * head_dim, fused.q_norm_weight, fused.eps,
                                   cos_row, sin_row, fused.rotary_dim, head_dim, fused_scratch[wave],
                                   [&](int d, float value) { dest[d] = float_to_bf16_bits(fused.q_row_scale ? value * q_factor : value); }, fused.interleaved);
            } else if (v == columns) {
                uint16_t* dest = k_pages + (((size_t)own_page * num_kv_heads + kvh) * PAGE + slot) * head_dim;
                norm_rotate_vector(projections + (size_t)(num_heads + kvh) * head_dim, fused.k_norm_weight, fused.eps, cos_row, sin_row,
                                   fused.rotary_dim, head_dim, fused_scratch[wave],
                                   [&](int d, float value) { dest[d] = float_to_bf16_bits(value); }, fused.interleaved);
            } else {
                const float* value = projections + (size_t)(num_heads + num_kv_heads) * head_dim + (size_t)kvh * v_dim;
                uint16_t* dest = v_pages + ((size_t)own_page * num_kv_heads + kvh) * v_dim * PAGE + slot;
                for (int d = lane; d < v_dim; d += 64) dest[(size_t)d * PAGE] = float_to_bf16_bits(value[d]);
            }
        }
        // the page is read below by this workgroup's own waves: its stores have to be done first
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        load_query<HD>(c, fused_q[valid ? col : 0], head_dim, valid);
    } else {
        load_query<HD>(c, q + ((size_t)row * num_heads + head) * head_dim, head_dim, valid);
    }
    // this lane's column is a head: its slope of a bias by distance, in the units of the raw scores
    float dist[1] = {slopes ? slopes[head] * 1.4426950408889634f / scale_log2 : 0.0f};
    if constexpr (STREAMED) {
#pragma unroll
        for (int i = 0; i < STAGES; ++i)
            if (own_round == i) {
                ask_for_keys(pages[i], offsets, keys_at(first_page[i], true));
                ask_for_values(pages[i], offsets, values_at(first_page[i], true));
                // waited for here: a wait in the loop that also allowed for this branch would hold up every round
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                    for (int dc = 0; dc < HD / 32; ++dc) asm volatile("" : "+v"(pages[i].k[kt][dc]));
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int t = 0; t < HD / 16; ++t) asm volatile("" : "+v"(pages[i].v[kb][t]));
            }
        for (int round = 0; round < my_rounds; round += STAGES) {
#pragma unroll
            for (int i = 0; i < STAGES; ++i) {
                if (round + i >= my_rounds) break;
                const int base = block_of(round + i) * PAGE;
                const bool wanted = round + i + STAGES < my_rounds;
                const int page = __builtin_amdgcn_readfirstlane(next[i]);
                // a lane without a head computes along (q = 0, nothing of it is stored)
                attend_on_way<HD>(c, pages[i], scale_log2, first - base, pos - base, cap, cap_scale, keep_first - base, slopes != nullptr, dist[0],
                                  [&] {
                                      next[i] = number_of(round + i + 2 * STAGES);
                                      ask_for_keys(pages[i], offsets, keys_at(page, wanted));
                                  },
                                  [&] { ask_for_values(pages[i], offsets, values_at(page, wanted)); });
            }
        }
    } else {
        for (int round = 0; round < my_rounds; ++round) {
            const int block = block_of(round), base = block * PAGE;
            const size_t at = ((size_t)number_of(round) * num_kv_heads + kvh) * PAGE;
            attend_page<HD, 1, true, false>(columns_of_wave, k_pages + at * head_dim, v_pages + at * v_dim, head_dim, v_dim, scale_log2, first - base, pos - base, pos - base,
                                            head_dim, PAGE, cap, cap_scale, keep_first - base, slopes ? dist : nullptr);
        }
    }
    const float l = fw_quad_sum(c.l);
#pragma unroll
    for (int t = 0; t < HD / 16; ++t) shared_o[wave][t][lane] = c.o[t];
    if (g == 0) {
        shared_m[wave][col] = c.m;
        shared_l[wave][col] = l;
    }
    __syncthreads();
    // how many workgroups work on this row: those whose first page holds a visible key
    const int row_splits = (last_step + 1 + pages_per_split - 1) / pages_per_split;
    // the sink of a head: one more part of the row, with maximum sink, sum 1 and no output (in units of log2)
    const float LOG2E_F = 1.4426950408889634f;
    const int stride = PART_STRIDE(v_dim);
    if (valid) {        // every wave: the four share out the channel tiles, each storing a quarter of the workgroup's result
        float m = NEG_BIG;
#pragma unroll
        for (int w = 0; w < SPLIT_PAGES; ++w) m = fmaxf(m, shared_m[w][col]);
        const bool final_here = row_splits == 1;
        const float sink = (sinks && final_here) ? sinks[head] * LOG2E_F : NEG_BIG;
        m = fmaxf(m, sink);
        float total = (sinks && final_here) ? exp2f(sink - m) : 0.0f, weight[SPLIT_PAGES];
#pragma unroll
        for (int w = 0; w < SPLIT_PAGES; ++w) {
            weight[w] = exp2f(shared_m[w][col] - m);        // a wave without a page has l = 0 and o = 0
            total += weight[w] * shared_l[w][col];
        }
        float* dest = partial + (((size_t)row * num_heads + head) * max_splits + split) * stride;
        uint16_t* final_dest = out + ((size_t)row * num_heads + head) * v_dim;
#pragma unroll
        for (int tt = 0; tt < (HD / 16 + SPLIT_PAGES - 1) / SPLIT_PAGES; ++tt) {
            const int t = tt * SPLIT_PAGES + wave;
            if (t >= HD / 16 || t * 16 >= v_dim) break;
            f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < SPLIT_PAGES; ++w) sum += weight[w] * shared_o[w][t][lane];
            if (row_splits == 1) {
                // the only workgroup of its row: the result is final
                const float inv = 1.0f / total;
                u32x2 packed = {pack_bf16(sum[0] * inv, sum[1] * inv), pack_bf16(sum[2] * inv, sum[3] * inv)};
                *reinterpret_cast<u32x2*>(final_dest + t * 16 + g * 4) = packed;
            } else {
                // device-scope stores: they pass the caches that workgroups on other dies do not share
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    __hip_atomic_store(dest + t * 16 + g * 4 + r, sum[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        if (wave == 0 && g == 0 && row_splits > 1) {
            __hip_atomic_store(dest + v_dim, m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(dest + v_dim + 1, total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if (row_splits == 1) return;
    // The workgroup of a (row, kv head) that arrives last merges the parts, in the order of the keys:
    // every wave waits for its own stores to be acknowledged, the workgroup meets, one thread
    // takes the ticket. Nobody waits for another workgroup. The ticket counter is left at zero.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int* ticket = tickets + (size_t)row * acrosses + across;
    if (threadIdx.x == 0) ticket_shared = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (ticket_shared != row_splits - 1) return;
    if (threadIdx.x == 0) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int columns = group - head_tile * 16 < 16 ? group - head_tile * 16 : 16;
    if (row_splits <= MERGE_PARTS && columns * v_dim > 2 * 64 * SPLIT_PAGES) {
        // More than two outputs a thread (many heads on one kv head, or wide values) and up to MERGE_PARTS parts: a thread per head first forms the parts' weights (their maxima and sums asked
        // for together, the weights kept in LDS), then every thread sums its outputs with many loads in flight:
        // eight outputs by eight parts at a time. With many heads on one kv head (hundreds of outputs a thread)
        // the walk below, one output after the other with each part's maximum and sum read again, took longer
        // than the attention itself. The parts are added in the order of the keys. (With one or two outputs a thread
        // the walk is one or two trips to memory and this would be three: a step of 8 rows with four heads of 64
        // channels to a kv head took 19.5 us this way against 17.0.)
        if (threadIdx.x < columns) {
            const float* source = partial + ((size_t)row * num_heads + kvh * group + head_tile * 16 + threadIdx.x) * max_splits * stride;
            float m = NEG_BIG;
            for (int sp0 = 0; sp0 < row_splits; sp0 += 8) {
                float ms[8], ls[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int sp = sp0 + u < row_splits ? sp0 + u : row_splits - 1;
                    ms[u] = __hip_atomic_load(source + (size_t)sp * stride + v_dim, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    ls[u] = __hip_atomic_load(source + (size_t)sp * stride + v_dim + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (sp0 + u < row_splits) {
                        merge_w[sp0 + u][threadIdx.x] = ms[u];
                        merge_l[sp0 + u][threadIdx.x] = ls[u];
                        m = fmaxf(m, ms[u]);
                    }
            }
            float total = 0.0f;
            if (sinks) {
                const float sink = sinks[kvh * group + head_tile * 16 + threadIdx.x] * LOG2E_F;
                m = fmaxf(m, sink);
                total = exp2f(sink - m);
            }
            for (int sp = 0; sp < row_splits; ++sp) {
                const float weight = exp2f(merge_w[sp][threadIdx.x] - m);
                total += weight * merge_l[sp][threadIdx.x];
                merge_w[sp][threadIdx.x] = weight;
            }
            merge_l[0][threadIdx.x] = 1.0f / total;
        }
        __syncthreads();
        const int items = columns * v_dim;
        for (int item0 = threadIdx.x; item0 < items; item0 += 64 * SPLIT_PAGES * 8) {
            float acc[8];
            const float* source[8];
            int column[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int item = item0 + 64 * SPLIT_PAGES * u < items ? item0 + 64 * SPLIT_PAGES * u : items - 1;
                column[u] = item / v_dim;
                source[u] = partial + ((size_t)row * num_heads + kvh * group + head_tile * 16 + column[u]) * max_splits * stride + item % v_dim;
                acc[u] = 0.0f;
            }
            for (int sp0 = 0; sp0 < row_splits; sp0 += 8) {
                float vs[8][8];
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const int sp = sp0 + q < row_splits ? sp0 + q : row_splits - 1;
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        vs[u][q] = __hip_atomic_load(source[u] + (size_t)sp * stride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    if (sp0 + q < row_splits) {
#pragma unroll
                        for (int u = 0; u < 8; ++u) acc[u] += merge_w[sp0 + q][column[u]] * vs[u][q];
                    }
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int item = item0 + 64 * SPLIT_PAGES * u;
                if (item < items)
                    out[((size_t)row * num_heads + kvh * group + head_tile * 16 + column[u]) * v_dim + item % v_dim] =
                        float_to_bf16_bits(acc[u] * merge_l[0][column[u]]);
            }
        }
        return;
    }
    for (int item = threadIdx.x; item < columns * v_dim; item += 64 * SPLIT_PAGES) {
        const int merged_head = kvh * group + head_tile * 16 + item / v_dim, d = item % v_dim;
        const float* source = partial + ((size_t)row * num_heads + merged_head) * max_splits * stride;
        // Sixteen parts are requested at a time (past the last one: the last one again, not used),
        // maximum, weight and value together: one round trip for up to sixteen parts. The running
        // sums are rescaled when a later batch of parts raises the maximum.
        auto part_at = [&](int sp, int offset) {
            const int clamped = sp < row_splits ? sp : row_splits - 1;
            return __hip_atomic_load(source + (size_t)clamped * stride + offset, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        };
        constexpr int AT_ONCE = 16;
        float m = NEG_BIG, total = 0.0f, acc = 0.0f;
        if (sinks) {
            m = sinks[merged_head] * LOG2E_F;
            total = 1.0f;
        }
        for (int sp0 = 0; sp0 < row_splits; sp0 += AT_ONCE) {
            float ms[AT_ONCE], ls[AT_ONCE], vs[AT_ONCE];
#pragma unroll
            for (int u = 0; u < AT_ONCE; ++u) {
                ms[u] = part_at(sp0 + u, v_dim);
                ls[u] = part_at(sp0 + u, v_dim + 1);
                vs[u] = part_at(sp0 + u, d);
            }
            float highest = m;
#pragma unroll
            for (int u = 0; u < AT_ONCE; ++u) highest = fmaxf(highest, ms[u]);
            const float keep = exp2f(m - highest);      // 0 for the first batch, whose sums are 0 anyway
            total *= keep;
            acc *= keep;
            m = highest;
#pragma unroll
            for (int u = 0; u < AT_ONCE; ++u) {
                const float weight = sp0 + u < row_splits ? exp2f(ms[u] - m) : 0.0f;
                total += weight * ls[u];
                acc += weight * vs[u];
            }
        }
        out[((size_t)row * num_heads + merged_head) * v_dim + d] = float_to_bf16_bits(acc / total);
    }
}

static const float LOG2E = 1.4426950408889634f;

// What the mask and the soft cap hand to the kernels: with a cap the scores are scaled and capped before
// the softmax, whose exponent then takes log2(e) alone.
struct ScoreRule {
    float scale_log2, cap, cap_scale;
};
static ScoreRule score_rule(float scale, float softcap) {
    if (softcap > 0.0f) return ScoreRule{LOG2E, softcap, scale / softcap};
    return ScoreRule{scale * LOG2E, 0.0f, 0.0f};
}
// the most keys a row can see where a window or a chunk bounds them (0: all)
static int visible_span(int window, int chunk) {
    int span = window;
    if (chunk > 0 && (span == 0 || chunk < span)) span = chunk;
    return span;
}

static int check_common(const char* name, int rows, int num_heads, int num_kv_heads, int head_dim, int v_dim, int page_size,
                        int window, int num_pages, int table_stride, int chunk = 0, float softcap = 0.0f) {
    FW_REQUIRE(chunk >= 0 && softcap >= 0.0f, "%s: chunk %d and soft cap %g must not be negative", name, chunk, (double)softcap);
    FW_REQUIRE(rows >= 0 && num_heads > 0 && num_kv_heads > 0 && num_heads % num_kv_heads == 0,
               "%s: heads %d must be a positive multiple of kv heads %d", name, num_heads, num_kv_heads);
    FW_REQUIRE(head_dim >= 16 && head_dim <= 256 && head_dim % 16 == 0, "%s: head_dim %d must be a multiple of 16 in 16..256", name, head_dim);
    FW_REQUIRE(v_dim >= 16 && v_dim <= 256 && v_dim % 16 == 0, "%s: the values' size %d must be a multiple of 16 in 16..256", name, v_dim);
    FW_REQUIRE(page_size == PAGE, "%s: page size must be %d, got %d", name, PAGE, page_size);
    FW_REQUIRE(window >= 0, "%s: window must be 0 (all keys) or positive, got %d", name, window);
    FW_REQUIRE(num_pages > 0 && table_stride > 0, "%s: empty cache (pages=%d, table stride=%d)", name, num_pages, table_stride);
    return 0;
}

#define FW_BY_HEAD_DIM(head_dim, CALL)      \
    do {                                    \
        if (head_dim <= 32) { CALL(32); }   \
        else if (head_dim <= 64) { CALL(64); } \
        else if (head_dim <= 128) { CALL(128); } \
        else { CALL(256); }                 \
    } while (0)

// bfloat16 q [rows][heads * head_dim] -> out (same shape). tile_seg / tile_row0 [tiles]: tiles of
// up to 64 rows that never span two segments, in any order (workgroups start in that order: list
// the tiles that see the most keys first). heads_together: query heads of a kv group that one
// workgroup takes (1, or 4 up to head_dim 64). Four read a page once for four heads (1.09 vs
// 1.27 ms for 2,048 rows behind 30,720 tokens, 32 heads in 8 groups, head_dim 64), one gives four
// times as many workgroups to even out tiles of unequal length (58 vs 81 us for the same rows
// from position 0; equal behind 6,144 tokens). The caller, who knows the positions, says which;
// 0: one. halves: 1 as above (PARTS 2 of the kernel for any head size), 2 heads two by two (attention_prompt_kernel), 3 those with the pages
// shared out between two halves.
extern "C" int fw_attention_prefill(const void* q, void* out, const void* k_pages, const void* v_pages,
                                    const int32_t* block_table, int table_stride, const int32_t* tile_seg,
                                    const int32_t* tile_row0, int tiles, const int32_t* seg_row0,
                                    const int32_t* row_pos, int rows, int num_heads, int num_kv_heads, int head_dim,
                                    int v_dim, float scale, int window, int chunk, float softcap, int keep_first, const float* sinks,
                                    const float* slopes, int page_size, int num_pages, int heads_together, int halves, void* stream) {
    FW_REQUIRE(keep_first >= 0 && (keep_first == 0 || chunk == 0), "attention_prefill: %d first keys are kept beside a window, not beside chunks", keep_first);
    if (check_common("attention_prefill", rows, num_heads, num_kv_heads, head_dim, v_dim, page_size, window, num_pages, table_stride, chunk, softcap)) return -1;
    const ScoreRule rule = score_rule(scale, softcap);
    const int widest = head_dim > v_dim ? head_dim : v_dim;      // the template holds both
    FW_REQUIRE(tiles >= 0 && tiles <= rows && num_heads <= 65535, "attention_prefill: %d tiles for %d rows", tiles, rows);
    const int most_together = widest <= 64 ? 4 : 1;
    FW_REQUIRE(heads_together == 0 || heads_together == 1 || (heads_together == 4 && most_together == 4),
               "attention_prefill: %d heads together with head_dim %d (1, or 4 up to head_dim 64)", heads_together, head_dim);
    FW_REQUIRE(halves >= 0 && halves <= 3, "attention_prefill: halves %d", halves);
    FW_REQUIRE(halves != 1 || (widest <= 64 && heads_together == 0), "attention_prefill: the pages are shared out between halves up to head_dim 64, two heads together");
    if (rows == 0 || tiles == 0) return 0;
    const int group = num_heads / num_kv_heads;
    const bool paired = halves >= 2;
    FW_REQUIRE(!paired || (heads_together == 0 && head_dim == v_dim && (head_dim == 64 || head_dim == 128) && group % 2 == 0),
               "attention_prefill: heads two by two are taken with head_dim and v_dim 64 or 128 and an even number of heads a group");
    if (halves) heads_together = 2;
    if (heads_together == 0) heads_together = 1;
    const long long blocks = (long long)tiles * num_kv_heads * ((group + heads_together - 1) / heads_together);
    FW_REQUIRE(blocks < (1ll << 31), "attention_prefill: too many tiles and heads");
    dim3 grid((unsigned)blocks);
#define LAUNCH_PROMPT(HD, PARTS, STG)                                                                               \
    {                                                                                                              \
        const int stage_bytes = PARTS * 2 * STG * PAGE * HD * 2, merge_bytes = PARTS > 1 ? 2 * (HD / 4 + 2) * 256 * 4 : 0;  \
        const int bytes = stage_bytes > merge_bytes ? stage_bytes : merge_bytes;                                   \
        static bool configured = false;                                                                            \
        if (!configured) {                                                                                         \
            hipError_t status = hipFuncSetAttribute((const void*)attention_prompt_kernel<HD, PARTS, STG>,          \
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, bytes);            \
            FW_REQUIRE(status == hipSuccess, "attention_prefill: cannot reserve %d bytes of LDS", bytes);          \
            configured = true;                                                                                     \
        }                                                                                                          \
        attention_prompt_kernel<HD, PARTS, STG><<<grid, 256 * PARTS, bytes, (hipStream_t)stream>>>(                 \
            (const uint16_t*)q, (uint16_t*)out, (const uint16_t*)k_pages, (const uint16_t*)v_pages, block_table,    \
            table_stride, tile_seg, tile_row0, seg_row0, row_pos, num_heads, num_kv_heads, rule.scale_log2,        \
            window, chunk, rule.cap, rule.cap_scale, keep_first, sinks, slopes);                                   \
    }
#define LAUNCH(HD, NH, PARTS)                                                                                      \
    {                                                                                                              \
        const int lds_bytes = PARTS * 2 * (PAGE * (HD + KV_PAD) + v_dim * (PAGE + KV_PAD)) * 2;                    \
        const int merge_bytes = PARTS > 1 ? NH * (HD / 4 + 2) * 256 * 4 : 0;                                       \
        const int bytes = lds_bytes > merge_bytes ? lds_bytes : merge_bytes;                                       \
        static int configured = 0;                                                                                 \
        if (bytes > configured) {                                                                                  \
            hipError_t status = hipFuncSetAttribute((const void*)attention_prefill_kernel<HD, NH, PARTS>,          \
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, bytes);            \
            FW_REQUIRE(status == hipSuccess, "attention_prefill: cannot reserve %d bytes of LDS", bytes);          \
            configured = bytes;                                                                                    \
        }                                                                                                          \
        attention_prefill_kernel<HD, NH, PARTS><<<grid, 256 * PARTS, bytes, (hipStream_t)stream>>>(                 \
            (const uint16_t*)q, (uint16_t*)out, (const uint16_t*)k_pages, (const uint16_t*)v_pages, block_table,    \
            table_stride, tile_seg, tile_row0, seg_row0, row_pos, num_heads, num_kv_heads, head_dim, v_dim,        \
            rule.scale_log2, window, chunk, rule.cap, rule.cap_scale, keep_first, sinks, slopes);                  \
    }
    if (paired) {
        if (head_dim == 64) {
            if (halves == 3) LAUNCH_PROMPT(64, 2, 4) else LAUNCH_PROMPT(64, 1, 4)
        } else {
            if (halves == 3) LAUNCH_PROMPT(128, 2, 2) else LAUNCH_PROMPT(128, 1, 2)
        }
    } else if (widest <= 32) {
        if (halves) LAUNCH(32, 2, 2) else if (heads_together == 4) LAUNCH(32, 4, 1) else LAUNCH(32, 1, 1)
    } else if (widest <= 64) {
        if (halves) LAUNCH(64, 2, 2) else if (heads_together == 4) LAUNCH(64, 4, 1) else LAUNCH(64, 1, 1)
    } else if (widest <= 128) {
        LAUNCH(128, 1, 1)
    } else {
        LAUNCH(256, 1, 1)
    }
#undef LAUNCH
#undef LAUNCH_PROMPT
    FW_LAUNCH_CHECK("attention_prefill");
    return 0;
}

static int decode_check(int max_splits, int max_context, int* tickets, int tickets_len, int table_stride, int rows, int num_heads,
                        int num_kv_heads, int head_dim, int v_dim, int window, int page_size, int num_pages, int chunk, float softcap,
                        int keep_first = 0) {
    FW_REQUIRE(keep_first >= 0 && (keep_first == 0 || chunk == 0), "attention_decode: %d first keys are kept beside a window, not beside chunks", keep_first);
    if (check_common("attention_decode", rows, num_heads, num_kv_heads, head_dim, v_dim, page_size, window, num_pages, table_stride, chunk, softcap)) return -1;
    window = visible_span(window, chunk);       // below: what bounds the pages a row's keys lie in
    FW_REQUIRE(max_splits >= 1 && max_splits <= 65535, "attention_decode: max_splits %d outside 1..65535", max_splits);
    FW_REQUIRE(max_context >= 1, "attention_decode: max_context must be positive");
    int blocks = (max_context + PAGE - 1) / PAGE;
    if (window > 0 && (window + PAGE - 2) / PAGE + 1 + (keep_first + PAGE - 1) / PAGE < blocks)
        blocks = (window + PAGE - 2) / PAGE + 1 + (keep_first + PAGE - 1) / PAGE;
    FW_REQUIRE(max_splits * SPLIT_PAGES >= blocks, "attention_decode: %d splits of %d pages do not cover %d pages of context",
               max_splits, SPLIT_PAGES, blocks);
    FW_REQUIRE((max_context + PAGE - 1) / PAGE <= table_stride, "attention_decode: a context of %d tokens exceeds the block table (%d pages)",
               max_context, table_stride);
    const int head_tiles = (num_heads / num_kv_heads + 15) / 16;
    FW_REQUIRE(rows <= 1 << 20 && num_kv_heads * head_tiles <= 65535 && num_heads <= 65535, "attention_decode: grid too large");
    FW_REQUIRE(rows == 0 || max_splits == 1 || (tickets != nullptr && (long long)tickets_len >= (long long)rows * num_kv_heads * head_tiles),
               "attention_decode: %d rows need %d ticket counters", rows, rows * num_kv_heads * head_tiles);
    return 0;
}

static int decode_launch(const void* q, void* out, float* partial, int max_splits, const int32_t* decode_work, int* tickets, void* k_pages, void* v_pages,
                         const int32_t* block_table, int table_stride, const int32_t* row_seg, const int32_t* row_pos, int rows,
                         int num_heads, int num_kv_heads, int head_dim, int v_dim, float scale, int window, int chunk, float softcap,
                         const FusedProjections& fused, int keep_first, const float* sinks, const float* slopes, void* stream) {
    if (rows == 0) return 0;
    const ScoreRule rule = score_rule(scale, softcap);
    const int head_tiles = (num_heads / num_kv_heads + 15) / 16;
    // Workgroups go to the eight dies in turn: the heads of a row first, so that a long row is spread over the dies (rows first, a
    // step of 8 n rows puts all of a row on one die: 64 ragged rows of up to 2,900 keys, 32 heads in 8 groups 59.9 us against 56.1; in 16 groups 117 against 107).
    const bool heads_first = rows <= 65535;
    const int across = num_kv_heads * head_tiles;
    const dim3 grid(heads_first ? across : rows, heads_first ? rows : across, max_splits);
    const EvenSplits even = even_splits(rows, across, max_splits, visible_span(window, chunk), keep_first);

#define CALL(HD)                                                                                                              \
    if (fused.qkv)                                                                                                            \
        attention_decode_split_kernel<HD, true><<<grid, 64 * SPLIT_PAGES, 0, (hipStream_t)stream>>>(                          \
            (const uint16_t*)q, (uint16_t*)out, partial, tickets, (uint16_t*)k_pages, (uint16_t*)v_pages, block_table,        \
            table_stride, row_seg, row_pos, num_heads, num_kv_heads, head_dim, v_dim, rule.scale_log2, window, chunk, rule.cap, rule.cap_scale, max_splits, decode_work, fused, keep_first, sinks, slopes, heads_first, even); \
    else                                                                                                                      \
        attention_decode_split_kernel<HD, false><<<grid, 64 * SPLIT_PAGES, 0, (hipStream_t)stream>>>(                         \
            (const uint16_t*)q, (uint16_t*)out, partial, tickets, (uint16_t*)k_pages, (uint16_t*)v_pages, block_table,        \
            table_stride, row_seg, row_pos, num_heads, num_kv_heads, head_dim, v_dim, rule.scale_log2, window, chunk, rule.cap, rule.cap_scale, max_splits, decode_work, fused, keep_first, sinks, slopes, heads_first, even)
    FW_BY_HEAD_DIM((head_dim > v_dim ? head_dim : v_dim), CALL);
#undef CALL
    FW_LAUNCH_CHECK("attention_decode");
    return 0;
}

// One row per request. partial: float32 workspace of rows * heads * max_splits * (head_dim + 4).
// max_context: no row's position reaches it (the caller knows; the kernel cannot check);
// max_splits must cover the keys such a row sees, in runs of 4 pages. decode_work: null, or one
// int32 on the device: the runs of 4 pages that all the rows of the step see together (the sum over
// the rows of ceil((position + 1) / 256)), or, where the rows are equally long, the runs of the longest as a negative number; with it a workgroup
// takes as many runs as bring the step down to about as many workgroups as compute units (it changes how the work is shared out, not what is computed). tickets: rows * kv heads *
// ceil(group / 16) int32 counters, zero before the first call and left zero; calls that overlap on
// one device need their own (and their own workspace).
extern "C" int fw_attention_decode(const void* q, void* out, float* partial, int max_splits, int max_context,
                                   const int32_t* decode_work, int* tickets, int tickets_len, const void* k_pages,
                                   const void* v_pages, const int32_t* block_table, int table_stride,
                                   const int32_t* row_seg, const int32_t* row_pos, int rows, int num_heads,
                                   int num_kv_heads, int head_dim, int v_dim, float scale, int window, int chunk, float softcap,
                                   int keep_first, const float* sinks, const float* slopes, int page_size, int num_pages, void* stream) {
    if (decode_check(max_splits, max_context, tickets, tickets_len, table_stride, rows, num_heads, num_kv_heads, head_dim, v_dim, window,
                     page_size, num_pages, chunk, softcap, keep_first)) return -1;
    return decode_launch(q, out, partial, max_splits, decode_work, tickets, const_cast<void*>(k_pages), const_cast<void*>(v_pages), block_table,
                         table_stride, row_seg, row_pos, rows, num_heads, num_kv_heads, head_dim, v_dim, scale, window, chunk, softcap, FusedProjections{}, keep_first, sinks, slopes, stream);
}

// fw_attention_decode with the work of fw_qk_norm_rope_kv_write in front of it, in the same kernel:
// qkv float32 [rows][(heads + 2 kv heads) * head_dim] are the step's raw projections; the new keys and
// values are stored in their pages (write_kv 0: they are there already and only the queries are
// formed). Norm weights float32 [head_dim] or null, rotation tables float32 [rows][rotary_dim / 2]
// (null with rotary_dim 0). Results as the two kernels one after the other give them.
extern "C" int fw_attention_decode_fused(const float* qkv, const float* q_norm_weight, const float* k_norm_weight, float eps,
                                         const float* cos_table, const float* sin_table, int rotary_dim, int write_kv, void* out,
                                         float* partial, int max_splits, int max_context, const int32_t* decode_work, int* tickets, int tickets_len,
                                         void* k_pages, void* v_pages, const int32_t* block_table, int table_stride,
                                         const int32_t* row_seg, const int32_t* row_pos, int rows, int num_heads,
                                         int num_kv_heads, int head_dim, int v_dim, float scale, int window, int chunk, float softcap,
                                         int interleaved, int q_only, int keep_first, const float* sinks, const float* slopes,
                                         const float* q_row_scale, int page_size, int num_pages, void* stream) {
    if (decode_check(max_splits, max_context, tickets, tickets_len, table_stride, rows, num_heads, num_kv_heads, head_dim, v_dim, window,
                     page_size, num_pages, chunk, softcap, keep_first)) return -1;
    FW_REQUIRE(!(q_only && write_kv), "attention_decode_fused: rows that hold queries only bring no keys or values to store");
    FW_REQUIRE(qkv != nullptr, "attention_decode_fused: the projections are missing");
    FW_REQUIRE(rotary_dim >= 0 && rotary_dim <= head_dim && rotary_dim % 2 == 0, "attention_decode_fused: rotary_dim %d with head_dim %d",
               rotary_dim, head_dim);
    FW_REQUIRE(rotary_dim == 0 || (cos_table != nullptr && sin_table != nullptr), "attention_decode_fused: the rotation tables are missing");
    FW_REQUIRE((q_norm_weight == nullptr) == (k_norm_weight == nullptr), "attention_decode_fused: q and k are normed together or not at all");
    FusedProjections fused;
    fused.qkv = qkv; fused.q_norm_weight = q_norm_weight; fused.k_norm_weight = k_norm_weight; fused.eps = eps;
    fused.cos_table = cos_table; fused.sin_table = sin_table; fused.rotary_dim = rotary_dim; fused.write_kv = write_kv;
    fused.interleaved = interleaved;
    fused.q_row_scale = q_row_scale;
    fused.width = q_only ? num_heads * head_dim : (num_heads + num_kv_heads) * head_dim + num_kv_heads * v_dim;
    return decode_launch(nullptr, out, partial, max_splits, decode_work, tickets, k_pages, v_pages, block_table, table_stride, row_seg, row_pos,
                         rows, num_heads, num_kv_heads, head_dim, v_dim, scale, window, chunk, softcap, fused, keep_first, sinks, slopes, stream);
}
