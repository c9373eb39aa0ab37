// Attention of prompt portions over the paged cache on the exact 32-bit path: the same formula
// as attention_generic.hip (reference: fused_ops.rs:430-535), tiled so that the keys and values a
// block needs are read once for a tile of query tokens and all query heads of a key/value head.
//
// A block of four waves owns 16 query rows (32 where a token's heads are more): consecutive tokens of one request, all query
// heads of one key/value head.  Keys go by in blocks of 64 that are
// aligned to absolute key positions (block c holds keys 64 c .. 64 c + 63), so that what a query
// row adds up, and in which order, depends on its position alone and not on how the prompt was
// cut: dot products of head-size terms in ascending order, the row's maximum and sum over the block in a
// fixed tree, and the weighted sum over the 64 keys in ascending order.  All arithmetic is 32-bit: fused multiply-adds, on
// the 32-bit matrix instruction; nothing is rounded below that.
// Cache layout: keys [pages][Hkv][page][hd], values [pages][Hkv][hd][page].  hd % 4 == 0, hd <= 128.
//
// What a query row adds up, and in which order, is the same in all forms of the kernel (for
// prompt portions, for a token's keys in turn and for one block of them), so that a token's
// output has the same bits whether its step held prompt portions or not:
//   - a block of 64 keys gives the row a partial result of its own: the largest score m_b, the
//     probabilities exp(s - m_b), their sum l_b and the weighted values acc_b, each summed in
//     ascending order from zero;
//   - the partial results are merged in ascending order of the blocks (merge_block).
// Products and sums that must round the same way everywhere are written with fmaf, __fmul_rn and
// __fsub_rn, and contraction is switched off for the file.
#include "common.h"
#include <algorithm>
#include <math.h>

#pragma clang fp contract(off)

namespace {

constexpr int EX_ROWS = 32;      // query rows a block, at most
constexpr int EX_KEYS = 64;      // keys a step: one a lane

// Merge a block's partial result (m_b, l_b, acc_b) into the running one (m, l, acc).
template <int NC>
__device__ __forceinline__ void merge_block(float& m, float& l, float (&acc)[NC], float m_b, float l_b, const float (&acc_b)[NC]) {
    if (!(m_b > -INFINITY)) return;                    // the row saw no key of this block
    const float M = fmaxf(m, m_b);
    const float alpha = expf(__fsub_rn(m, M));         // 0 while nothing has been seen (m = -inf)
    const float beta = expf(__fsub_rn(m_b, M));
    l = fmaf(l, alpha, __fmul_rn(l_b, beta));
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = fmaf(acc[c], alpha, __fmul_rn(acc_b[c], beta));
    m = M;
}

typedef float exf32x4_t __attribute__((ext_vector_type(4)));

// Four registers of the four lane groups (lane / 16), transposed: register s of group g becomes register g of group s.
__device__ __forceinline__ void transpose_groups(float4& v) {
    uint32_t x0 = __float_as_uint(v.x), x1 = __float_as_uint(v.y), x2 = __float_as_uint(v.z), x3 = __float_as_uint(v.w);
    auto a = __builtin_amdgcn_permlane32_swap(x0, x2, false, false);
    auto b = __builtin_amdgcn_permlane32_swap(x1, x3, false, false);
    auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    v = make_float4(__uint_as_float(c[0]), __uint_as_float(c[1]), __uint_as_float(d[0]), __uint_as_float(d[1]));
}
__device__ __forceinline__ float elem(const float4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// v_mfma_f32_16x16x4_f32 gives D = A.B + C with the four products added to C one after the other, each a fused multiply-add
// rounded to 32 bits (denormals kept): the sums of an FMA loop over the same index, bit for bit, at twice its rate and with
// no operand read from LDS.
//
// A block owns RT tiles of 16 query rows on one key/value head; its four waves take a block of 64 keys together:
//   - scores: wave w multiplies keys 16 w .. 16 w + 15 with all rows.  Row m of the instruction's A holds key 4 (m % 4) + m / 4, so
//     that element i of lane group g of the result is key 4 i + g, which is where the second product wants it.  A lane reads four
//     consecutive features of its key; transpose_groups makes them the four steps' operands.
//   - the waves' maxima meet in LDS, then their probabilities (two barriers a block of keys, two buffers of each); every wave
//     reads all 64 of its lanes' rows and makes their sum itself, whose tree is that of wave_sum over a lane a key.
//   - weighted values: wave w makes the features 16 w .. 16 w + 15 (and those 64 on), keys in ascending order.
// Keys, values and page ids are asked for a block of keys ahead.  SINGLE: a block's rows are one token's heads.
// What bounds it: the chain of a block of keys (16 dependent matrix instructions, two barriers, exponentials, 16 more), about 1.7 us
// where a unit holds one block, and the instructions beside the matrix instructions where it holds four.  Measured, us, with FMAs on
// operands from LDS (and a key a lane for single tokens) before / now, 32 heads, 8 of keys: 600 tokens at head 64 151 / 45, 100 tokens 31 / 7.5,
// 2,048 tokens 1024 / 327 (52 TFLOP/s), 64 tokens behind 2,000 544 / 66, 7 single tokens behind 1,500 beside 64 more 416 / 52; head 128:
// 600 tokens 471 / 84; 2,048 tokens of 24 heads 2748 / 504.
constexpr uint32_t EX_FEW_BLOCKS = 2048;               // up to so many, the chip holds half of them at once
enum { EX_PORTIONS = 0, EX_SINGLE = 1, EX_BLOCKS = 2, EX_RANGES = 3 };
template <int NJ, int RT, int MODE, bool ANY>          // NJ: groups of 16 features, 4 or 8; ANY: pages of any size, else of 2^page_shift >= 4
__global__ __launch_bounds__(256, NJ * RT > 4 ? 2 : 4) void attn_exact_f32_kernel(
        const float* __restrict__ q, int q_stride, float* __restrict__ out, int out_stride,
        const float* __restrict__ kc, const float* __restrict__ vc,
        const int* __restrict__ table, int max_blocks,
        const int* __restrict__ cu_q, const int* __restrict__ q_start, const int* __restrict__ row_of_token,
        const int* __restrict__ positions, const int* __restrict__ kv_lens,
        int num_rows, int H, int Hkv, int hd, int page, int page_shift, float scale, int window, int TQ,
        int slots, int range, float* __restrict__ part_ml, float* __restrict__ part_o) {
    constexpr int NF = NJ / 4;                         // feature tiles a wave
    constexpr bool PARTIAL = MODE == EX_BLOCKS || MODE == EX_RANGES;       // every block of keys leaves a partial result
    __shared__ float4 probs[2][RT][4][64];             // [buffer][row tile][key tile][lane]
    __shared__ float tops[2][RT][4][16];               // [buffer][row tile][key tile][row]
    const int g_kv = blockIdx.y, G = H / Hkv;
    int b = -1, t0 = 0, nt = 0, p0 = 0;
    if (MODE != EX_PORTIONS) {
        t0 = MODE == EX_SINGLE ? blockIdx.x : blockIdx.z;
        nt = 1;
        b = row_of_token[t0];
        p0 = positions[t0];
        // a padding token, or behind the token, as most blocks of a large step are: gone after one trip to memory (which costs the others 0.5 us)
        if (PARTIAL && gridDim.x * gridDim.y * gridDim.z > EX_FEW_BLOCKS && (b < 0 || ((window > 0 ? max(0, p0 + 1 - window) : 0) / EX_KEYS + (int)blockIdx.x * (MODE == EX_BLOCKS ? 1 : range)) * EX_KEYS > p0)) return;
    } else {
        // which request and which of its tokens: tiles are numbered request by request; late tiles, which see the most keys, run first
        const int tile = (int)gridDim.x - 1 - (int)blockIdx.x;
        int before = 0;
        for (int r = 0; r < num_rows; ++r) {
            const int lo = cu_q[r], ql = cu_q[r + 1] - lo, tiles = (ql + TQ - 1) / TQ;
            if (tile < before + tiles) {
                b = r;
                t0 = lo + (tile - before) * TQ;
                nt = min(TQ, lo + ql - t0);
                break;
            }
            before += tiles;
        }
        if (b < 0) return;
        p0 = q_start[b] + (t0 - cu_q[b]);              // position of the tile's first token
    }
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int R = nt * G;                              // rows in use: row i = token i / G, head i % G of the group
    const int kv_len = b >= 0 ? kv_lens[b] : 0;        // a padding token sees nothing
    const int last_visible = min(kv_len, p0 + nt);     // of the tile's last token
    const int first_key = window > 0 ? max(0, p0 + 1 - window) : 0;   // of its first
    const int* pages = table + (size_t)max(b, 0) * max_blocks;
    auto page_of = [&](int key) { return (uint32_t)(ANY ? key / page : key >> page_shift); };
    auto slot_of = [&](int key) { return ANY ? key % page : key & (page - 1); };
    const uint32_t page_size = (uint32_t)Hkv * page * hd;                     // values of a page
    const float* kg = kc + (size_t)g_kv * page * hd;
    const float* vg = vc + (size_t)g_kv * page * hd;

    float4 qt[RT][NJ];                                 // .x .. .w: features 16 j + 4 s + g of the lane's row
    int row_lo[RT], row_hi[RT];                        // keys [row_lo, row_hi) are the row's
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int i = rt * 16 + r, p = p0 + i / G;
        row_hi[rt] = i < R ? min(kv_len, p + 1) : 0;
        row_lo[rt] = window > 0 ? max(0, p + 1 - window) : 0;
        const float* qr = q + (size_t)(t0 + (i < R ? i / G : 0)) * q_stride + (size_t)(g_kv * G + (i < R ? i % G : 0)) * hd;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            const int d = 16 * j + 4 * g;
            if (i < R && d < hd) v = make_float4(qr[d], qr[d + 1], qr[d + 2], qr[d + 3]);
            transpose_groups(v);
            qt[rt][j] = v;
        }
    }
    float m[RT], l[RT];
    exf32x4_t acc[RT][NF];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        m[rt] = -INFINITY;
        l[rt] = 0.f;
#pragma unroll
        for (int f = 0; f < NF; ++f) acc[rt][f] = exf32x4_t{0.f, 0.f, 0.f, 0.f};
    }

    // The lane's key of a block's tile w, and its four keys of each tile of values.  Every load is made, from the last visible
    // key or from page 0 where there is none to make, and what it brings is put to zero where it is used: loads under a
    // condition would be waited for all at once.
    const int kj = 16 * wave + 4 * (r & 3) + (r >> 2);
    int kb0 = first_key / EX_KEYS, kb1 = last_visible > first_key ? (last_visible + EX_KEYS - 1) / EX_KEYS : kb0;
    const int kb_first = kb0;                          // of the token: slot 0 of its partial results
    if (PARTIAL) {                                     // one block of keys, or `range` of them in turn
        kb0 += (int)blockIdx.x * (MODE == EX_BLOCKS ? 1 : range);
        kb1 = min(kb1, kb_first + slots);              // whatever kv_lens says
        if (kb0 >= kb1) return;
        kb1 = MODE == EX_BLOCKS ? kb0 + 1 : min(kb1, kb0 + range);
    }
    int pk = -1, pv[4] = {-1, -1, -1, -1};             // pages of the block that is asked for next
    bool v_there[4] = {};                              // of the block that is used next
    auto ask_pages = [&](int kb) {
        pk = pages[page_of(min(kb * EX_KEYS + kj, last_visible - 1))];
        if (!ANY)
#pragma unroll
            for (int t = 0; t < 4; ++t) pv[t] = pages[page_of(min(kb * EX_KEYS + 16 * t + 4 * g, last_visible - 1))];
    };
    float4 kt[NJ], vt[NF][4];
    auto ask_keys = [&](int kb) {                      // where there is no key: its score is not looked at
        const float* kr = kg + (size_t)(uint32_t)max(pk, 0) * page_size + (uint32_t)slot_of(kb * EX_KEYS + kj) * (uint32_t)hd;
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj) {
            const int d = 16 * jj + 4 * g;
            kt[jj] = *reinterpret_cast<const float4*>(kr + (d < hd ? d : 0));
        }
    };
    auto ask_values = [&](int kb) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int key = kb * EX_KEYS + 16 * t + 4 * g;
            if (!ANY) {
                v_there[t] = pv[t] >= 0;
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    const int d = min(16 * (wave + 4 * f) + r, hd - 1);
                    vt[f][t] = *reinterpret_cast<const float4*>(vg + (size_t)(uint32_t)max(pv[t], 0) * page_size + (uint32_t)(d * page + slot_of(key)));
                }
            } else {
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    const int d = min(16 * (wave + 4 * f) + r, hd - 1);
                    float x[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const int pid = key + u < last_visible ? pages[page_of(key + u)] : -1;
                        x[u] = pid >= 0 ? vg[(size_t)(uint32_t)pid * page_size + (uint32_t)(d * page + slot_of(key + u))] : 0.f;
                    }
                    vt[f][t] = make_float4(x[0], x[1], x[2], x[3]);
                }
            }
        }
    };
    if (kb0 < kb1) {
        ask_pages(kb0);
        ask_keys(kb0);
        ask_values(kb0);
        if (MODE != EX_BLOCKS) ask_pages(min(kb0 + 1, kb1 - 1));
    }
    for (int kb = kb0; kb < kb1; ++kb) {
        const int j_base = kb * EX_KEYS, buf = kb & 1;
        const int next = min(kb + 1, kb1 - 1);
        exf32x4_t s[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) s[rt] = exf32x4_t{0.f, 0.f, 0.f, 0.f};
        float4 k4[NJ];
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj) {
            const uint32_t feature = 16 * jj + 4 * g < hd ? 0xffffffffu : 0u;          // (as a mask: no branch around the wait)
            k4[jj] = make_float4(__uint_as_float(__float_as_uint(kt[jj].x) & feature), __uint_as_float(__float_as_uint(kt[jj].y) & feature),
                                 __uint_as_float(__float_as_uint(kt[jj].z) & feature), __uint_as_float(__float_as_uint(kt[jj].w) & feature));
            transpose_groups(k4[jj]);
        }
        if (MODE != EX_BLOCKS) ask_keys(next);
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj)
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
                    s[rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(elem(k4[jj], u), elem(qt[rt][jj], u), s[rt], 0, 0, 0);
        // element i: key 16 w + 4 i + g of the block
        float sc[RT][4];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int j = j_base + 16 * wave + 4 * i + g;
                sc[rt][i] = j >= row_lo[rt] && j < row_hi[rt] ? __fmul_rn(s[rt][i], scale) : -INFINITY;
            }
            float top = fmaxf(fmaxf(sc[rt][0], sc[rt][1]), fmaxf(sc[rt][2], sc[rt][3]));
            top = fmaxf(top, __shfl_xor(top, 16, 64));
            top = fmaxf(top, __shfl_xor(top, 32, 64));
            if (g == 0) tops[buf][rt][wave][r] = top;
        }
        __syncthreads();
        float m_b[RT], l_b[RT];
        float4 p[RT][4];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            // a key that is not the row's has the score -inf and the probability zero, also where the row has no key here
            m_b[rt] = fmaxf(fmaxf(fmaxf(tops[buf][rt][0][r], tops[buf][rt][1][r]), fmaxf(tops[buf][rt][2][r], tops[buf][rt][3][r])), -INFINITY);
            const float top = m_b[rt] > -INFINITY ? m_b[rt] : 0.f;
            probs[buf][rt][wave][lane] = make_float4(expf(__fsub_rn(sc[rt][0], top)), expf(__fsub_rn(sc[rt][1], top)),
                                                     expf(__fsub_rn(sc[rt][2], top)), expf(__fsub_rn(sc[rt][3], top)));
        }
        __syncthreads();
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
            for (int t = 0; t < 4; ++t) p[rt][t] = probs[buf][rt][t][lane];
            // wave_sum's tree with key = 16 t + 4 i + g for the lane: t ^ 2, t ^ 1, i ^ 2, i ^ 1, g ^ 2, g ^ 1
            float e[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                e[i] = (elem(p[rt][0], i) + elem(p[rt][2], i)) + (elem(p[rt][1], i) + elem(p[rt][3], i));
            float sum = (e[0] + e[2]) + (e[1] + e[3]);
            sum += __shfl_xor(sum, 32, 64);
            sum += __shfl_xor(sum, 16, 64);
            l_b[rt] = sum;
        }
        exf32x4_t acc_b[RT][NF];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int f = 0; f < NF; ++f) acc_b[rt][f] = exf32x4_t{0.f, 0.f, 0.f, 0.f};
        float4 v4[NF][4];
        // the rest of a last page, and a page that the window has passed and given back, may hold anything
        const bool cut = !ANY && (j_base + EX_KEYS > last_visible || __any(!(v_there[0] && v_there[1] && v_there[2] && v_there[3])));
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int t = 0; t < 4; ++t) v4[f][t] = vt[f][t];
        if (cut) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int key = j_base + 16 * t + 4 * g, there = v_there[t] ? last_visible : 0;
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    v4[f][t].x = key < there ? v4[f][t].x : 0.f;
                    v4[f][t].y = key + 1 < there ? v4[f][t].y : 0.f;
                    v4[f][t].z = key + 2 < there ? v4[f][t].z : 0.f;
                    v4[f][t].w = key + 3 < there ? v4[f][t].w : 0.f;
                }
            }
        }
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int t = 0; t < 4; ++t) transpose_groups(v4[f][t]);
        if (MODE != EX_BLOCKS) {
            ask_values(next);
            ask_pages(min(kb + 2, kb1 - 1));
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int f = 0; f < NF; ++f)
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt)
                        acc_b[rt][f] = __builtin_amdgcn_mfma_f32_16x16x4f32(elem(v4[f][t], i), elem(p[rt][t], i), acc_b[rt][f], 0, 0, 0);
        if (PARTIAL) {                                 // the block's partial results
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const int i = rt * 16 + r;
                if (i >= R) continue;
                const size_t at = ((size_t)t0 * H + (size_t)g_kv * G + i) * slots + (kb - kb_first);
                if (wave == 0 && g == 0) {
                    part_ml[at * 2] = m_b[rt];
                    part_ml[at * 2 + 1] = l_b[rt];
                }
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    const int d = 16 * (wave + 4 * f) + 4 * g;         // hd % 4 == 0
                    if (d < hd) *reinterpret_cast<float4*>(part_o + at * hd + d) =
                        make_float4(acc_b[rt][f][0], acc_b[rt][f][1], acc_b[rt][f][2], acc_b[rt][f][3]);
                }
            }
            continue;
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            float add[NF * 4], sum[NF * 4];
#pragma unroll
            for (int f = 0; f < NF; ++f)
#pragma unroll
                for (int e = 0; e < 4; ++e) { add[f * 4 + e] = acc_b[rt][f][e]; sum[f * 4 + e] = acc[rt][f][e]; }
            merge_block<NF * 4>(m[rt], l[rt], sum, m_b[rt], l_b[rt], add);
#pragma unroll
            for (int f = 0; f < NF; ++f)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[rt][f][e] = sum[f * 4 + e];
        }
    }
    if (PARTIAL) return;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int i = rt * 16 + r;
        if (i >= R) continue;
        float* o = out + (size_t)(t0 + i / G) * out_stride + (size_t)(g_kv * G + i % G) * hd;
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int d = 16 * (wave + 4 * f) + 4 * g + e;
                if (d < hd) o[d] = l[rt] > 0.f ? acc[rt][f][e] / l[rt] : 0.f;
            }
    }
}

// ---------------------------------------------------------------------------
// Single tokens.  A block takes one block of 64 keys of a token ("flash decoding"; reference:
// crates/infer-backend-cuda/src/kernels/flash_attn_gqa/flash_attn_paged_decode.cu:75-337), or several in turn, and leaves their partial
// results, and a second kernel merges a row's partial results in ascending order of the blocks; of few keys a block takes
// all of its token's, and there is no second kernel (exact_split).
// Partial results: part_ml [T][H][slots][2] = (m_b, l_b), part_o [T][H][slots][hd]; slot s of a
// token is key block first_block + s, first_block = (first visible key) / 64.
// ---------------------------------------------------------------------------
// One wave per (token, head): the partial results of its key blocks, merged in ascending order.
template <int NC>
__global__ __launch_bounds__(64) void attn_exact_combine_kernel(
        const float* __restrict__ part_ml, const float* __restrict__ part_o,
        const int* __restrict__ row_of_token, const int* __restrict__ positions, const int* __restrict__ kv_lens,
        int H, int hd, int window, int slots, float* __restrict__ out, int out_stride) {
    const int t = blockIdx.y, h = blockIdx.x, lane = threadIdx.x;
    const int b = row_of_token[t];
    int n = 0;                                          // a padding token, or nothing to see: zeros
    if (b >= 0) {
        const int p = positions[t];
        const int visible = min(kv_lens[b], p + 1);
        const int j0 = window > 0 ? max(0, p + 1 - window) : 0;
        if (visible > j0) n = min((visible - 1) / EX_KEYS - j0 / EX_KEYS + 1, slots);
    }
    const float* ml = part_ml + ((size_t)t * H + h) * slots * 2;
    const float* po = part_o + ((size_t)t * H + h) * slots * hd;
    float m = -INFINITY, l = 0.f, acc[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = 0.f;
    // eight partial results are asked for at a time (the loads do not depend on the merging), then
    // merged one after the other
    for (int s0 = 0; s0 < n; s0 += 8) {
        float mb[8], lb[8], acc_b[8][NC];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int s = min(s0 + u, n - 1);
            mb[u] = s0 + u < n ? ml[2 * s] : -INFINITY;      // -inf: merge_block leaves everything as it is
            lb[u] = ml[2 * s + 1];
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const int d = lane + 64 * c;
                acc_b[u][c] = d < hd ? po[(size_t)s * hd + d] : 0.f;
            }
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) merge_block<NC>(m, l, acc, mb[u], lb[u], acc_b[u]);
    }
    float* o = out + (size_t)t * out_stride + (size_t)h * hd;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int d = lane + 64 * c;
        if (d < hd) o[d] = l > 0.f ? acc[c] / l : 0.f;
    }
}

// How a single token's keys are divided between blocks: `range` blocks of 64 keys a block, in turn, and `blocks` blocks a (token, key/value
// head) pair; range 0: all of them in one block that writes the output itself, with no merge.  The step is planned for a longest length that
// its rows need not have (a captured step for its bucket's), and rows differ: blocks beyond a row's end are as common as others, so they leave after
// one trip to memory, and a long row is not left to one block.  One block of keys a block while there are up to 30,000 blocks; above, ranges of 4 to 64.
// An odd number of blocks a pair: consecutive ones go around the eight XCDs, and the empty ones would all be some XCDs'.
// Measured, us, a key a lane and a wave a block of keys (first) / a block of keys a block, all of a token's from 512 pairs on (then) / now, 8 key/value heads
// of 64: 64 tokens, one of 16,000 keys and the others of 200 97 / 703 / 86, one of 3,000 and the others of 100 42 / 137 / 30; 64 ragged up to 1,000
// keys 51 / 52 / 30, up to 4,000 155 / 186 / 120, equal 1,000 95 / 54 / 64, 4,000 313 / 195 / 230; 16, one of 16,000 84 / 94 / 73; 128 tokens of 32
// heads of 128 with keys of their own, ragged up to 1,000 424 / 461 / 356, but up to 60 67 / 80 / 91.  (Equal rows lose what ragged ones need: no length but
// the longest is known here.)
constexpr int EX_SINGLE_KEYS = 128;
struct ExactSplit { int blocks, range; };
ExactSplit exact_split(long long pairs, int max_kv_len) {
    if (max_kv_len <= EX_SINGLE_KEYS) return {1, 0};
    const int slots = (max_kv_len + EX_KEYS - 1) / EX_KEYS + 1;           // a window may begin inside a block: one more
    const long long most = std::max(30000 / pairs, 1ll);
    const int range = most >= slots ? 1 : (int)std::min(std::max((slots + most - 1) / most, 4ll), 64ll);
    return {((slots + range - 1) / range) | 1, range};
}

// Two tiles of rows a block where a token's heads fill more than one, or values are read one at a time: pages of no power of two of four keys and
// more, or a value cache that does not begin at a multiple of 16 bytes (shift -1).
int exact_page_shift(int page, const float* vc) { return page >= 4 && (page & (page - 1)) == 0 && (uintptr_t)vc % 16 == 0 ? __builtin_ctz((unsigned)page) : -1; }
bool exact_two_tiles(int G, int shift) { return G > 16 || shift < 0; }

template <int MODE>
void launch_exact(dim3 grid, int hd, int TQ, const float* q, int q_stride, float* out, int out_stride, const float* kc, const float* vc,
                  const int* table, int max_blocks, const int* cu_q, const int* q_start, const int* row_of_token, const int* positions,
                  const int* kv_lens, int num_rows, int H, int Hkv, int page, float scale, int window, int slots, int range, float* part_ml, float* part_o,
                  hipStream_t stream) {
    const int shift = exact_page_shift(page, vc);
    const bool two = exact_two_tiles(H / Hkv, shift);
#define RI_EXACT(NJ_, RT_, ANY_) attn_exact_f32_kernel<NJ_, RT_, MODE, ANY_><<<grid, 256, 0, stream>>>(q, q_stride, out, out_stride, kc, vc, table, max_blocks, \
        cu_q, q_start, row_of_token, positions, kv_lens, num_rows, H, Hkv, hd, page, shift, scale, window, TQ, slots, range, part_ml, part_o)
    if (hd <= 64) { if (shift < 0) RI_EXACT(4, 2, true); else if (two) RI_EXACT(4, 2, false); else RI_EXACT(4, 1, false); }
    else { if (shift < 0) RI_EXACT(8, 2, true); else if (two) RI_EXACT(8, 2, false); else RI_EXACT(8, 1, false); }
#undef RI_EXACT
}

}  // namespace

// exact_split, for a test without a GPU.
extern "C" void ri_attention_exact_split(int T, int Hkv, int max_kv_len, int* blocks, int* range) {
    const ExactSplit split = exact_split((long long)T * Hkv, max_kv_len);
    *blocks = split.blocks;
    *range = split.range;
}

// Whether ri_attention_exact_f32 takes these sizes (else: the generic kernel).
extern "C" int ri_attention_exact_supported(int H, int Hkv, int hd, int page) {
    return H > 0 && Hkv > 0 && H % Hkv == 0 && H / Hkv <= EX_ROWS && hd > 0 && hd % 4 == 0 && hd <= 128 && page > 0;
}

// Every token of the step belongs to a request row (cu_q covers all T tokens); rows of one token
// are taken as well, but a step of single tokens only is better served by the entry point below,
// which spreads it over more blocks.
extern "C" int ri_attention_exact_f32(
        const float* q, int q_stride, float* out, int out_stride, const float* kc, const float* vc,
        int num_pages, int page, int H, int Hkv, int hd, const int* table, int max_blocks,
        const int* cu_q, const int* q_start, const int* kv_lens, int num_rows, int T,
        float scale, int window, hipStream_t stream) {
    RI_REQUIRE(ri_attention_exact_supported(H, Hkv, hd, page), "ri_attention_exact_f32: sizes not taken (H=%d Hkv=%d hd=%d page=%d)", H, Hkv, hd, page);
    RI_REQUIRE(T >= 0 && num_rows >= 0 && max_blocks > 0 && num_pages > 0 && window >= 0, "ri_attention_exact_f32: bad sizes");
    RI_REQUIRE(q_stride >= H * hd && out_stride >= H * hd, "ri_attention_exact_f32: row strides too small");
    if (T == 0 || num_rows == 0) return 0;
    RI_REQUIRE(q && out && kc && vc && table && cu_q && q_start && kv_lens, "ri_attention_exact_f32: null pointer");
    RI_REQUIRE((uintptr_t)kc % 16 == 0, "ri_attention_exact_f32: unaligned key cache");
    RI_REQUIRE(Hkv <= 65535, "ri_attention_exact_f32: too many key/value heads for the grid");
    const int G = H / Hkv;
    const int TQ = (exact_two_tiles(G, exact_page_shift(page, vc)) ? 32 : 16) / G;
    const int tiles = (T + TQ - 1) / TQ + num_rows;    // at most: every request may end in a short tile
    launch_exact<EX_PORTIONS>(dim3(tiles, Hkv), hd, TQ, q, q_stride, out, out_stride, kc, vc, table, max_blocks, cu_q, q_start, nullptr, nullptr, kv_lens,
                              num_rows, H, Hkv, page, scale, window, 0, 0, nullptr, nullptr, stream);
    RI_LAUNCHED("ri_attention_exact_f32");
    return 0;
}

// Floats of workspace ri_attention_exact_decode_f32 needs for T tokens whose longest request has
// max_kv_len keys.
extern "C" size_t ri_attention_exact_decode_workspace(int T, int H, int hd, int max_kv_len) {
    const size_t slots = (size_t)(max_kv_len + EX_KEYS - 1) / EX_KEYS + 1;
    return (size_t)T * H * slots * (hd + 2);
}

// A step of single tokens on the exact path (every row of the step has one token; padding tokens
// carry row -1).  Same sizes as ri_attention_exact_supported.  The output of a token has the bits
// that ri_attention_exact_f32 gives the same token as part of any step.
extern "C" int ri_attention_exact_decode_f32(
        const float* q, int q_stride, float* out, int out_stride, const float* kc, const float* vc,
        int num_pages, int page, int H, int Hkv, int hd, const int* table, int max_blocks,
        const int* row_of_token, const int* positions, const int* kv_lens, int T, int max_kv_len,
        float scale, int window, float* workspace, size_t workspace_floats, hipStream_t stream) {
    RI_REQUIRE(ri_attention_exact_supported(H, Hkv, hd, page), "ri_attention_exact_decode_f32: sizes not taken (H=%d Hkv=%d hd=%d page=%d)", H, Hkv, hd, page);
    RI_REQUIRE(T >= 0 && max_kv_len > 0 && max_blocks > 0 && num_pages > 0 && window >= 0, "ri_attention_exact_decode_f32: bad sizes");
    RI_REQUIRE(q_stride >= H * hd && out_stride >= H * hd && q_stride % 4 == 0, "ri_attention_exact_decode_f32: bad row strides");
    if (T == 0) return 0;
    RI_REQUIRE(q && out && kc && vc && table && row_of_token && positions && kv_lens && workspace, "ri_attention_exact_decode_f32: null pointer");
    RI_REQUIRE((uintptr_t)kc % 16 == 0 && (uintptr_t)vc % 16 == 0 && (uintptr_t)q % 16 == 0 && (uintptr_t)workspace % 16 == 0,
               "ri_attention_exact_decode_f32: unaligned operands");
    RI_REQUIRE(Hkv <= 65535 && T <= 65535 && H <= 65535, "ri_attention_exact_decode_f32: too many heads or tokens for the grid");
    RI_REQUIRE(workspace_floats >= ri_attention_exact_decode_workspace(T, H, hd, max_kv_len),
               "ri_attention_exact_decode_f32: workspace of %zu floats, %zu needed", workspace_floats,
               ri_attention_exact_decode_workspace(T, H, hd, max_kv_len));
    const ExactSplit split = exact_split((long long)T * Hkv, max_kv_len);
    if (split.range == 0) {
        launch_exact<EX_SINGLE>(dim3(T, Hkv), hd, 1, q, q_stride, out, out_stride, kc, vc, table, max_blocks, nullptr, nullptr, row_of_token, positions,
                                kv_lens, T, H, Hkv, page, scale, window, 0, 0, nullptr, nullptr, stream);
        RI_LAUNCHED("ri_attention_exact_decode_f32");
        return 0;
    }
    const int slots = (max_kv_len + EX_KEYS - 1) / EX_KEYS + 1;
    float* part_ml = workspace + (size_t)T * H * slots * hd;
    float* part_o = workspace;
    const dim3 grid(split.blocks, Hkv, T);
    if (split.range == 1)
        launch_exact<EX_BLOCKS>(grid, hd, 1, q, q_stride, out, out_stride, kc, vc, table, max_blocks, nullptr, nullptr, row_of_token, positions,
                                kv_lens, T, H, Hkv, page, scale, window, slots, 1, part_ml, part_o, stream);
    else
        launch_exact<EX_RANGES>(grid, hd, 1, q, q_stride, out, out_stride, kc, vc, table, max_blocks, nullptr, nullptr, row_of_token, positions,
                                kv_lens, T, H, Hkv, page, scale, window, slots, split.range, part_ml, part_o, stream);
    RI_LAUNCHED("ri_attention_exact_decode_f32");
    auto combine = hd <= 64 ? attn_exact_combine_kernel<1> : attn_exact_combine_kernel<2>;
    combine<<<dim3(H, T), 64, 0, stream>>>(part_ml, part_o, row_of_token, positions, kv_lens, H, hd, window, slots, out, out_stride);
    RI_LAUNCHED("ri_attention_exact_decode_f32(combine)");
    return 0;
}
