// bfloat16 attention of single tokens over the paged cache on the matrix cores (gfx950),
// with the key range split over waves ("flash decoding"; reference:
// crates/infer-backend-cuda/src/kernels/flash_attn_gqa/flash_attn_paged_decode.cu:75-337).
//
// One wave per (chunk of 64 or 128 keys, kv head, token); for long contexts a wave takes several
// chunks, one after the other, with a running maximum and sum, so that the number of partial
// results stays bounded.  All query heads of the kv head share each key and value load (they are the 16 columns of the MFMA tiles, G = H/Hkv <= 16 used).
//   S^T[key, q]  = K_tile[16 keys, hd] . Q^T[hd, 16 q]        v_mfma_f32_16x16x32_bf16
//   P^T = exp(S^T * scale - max)                                 in registers, 32-bit
//   O[q, d]     += P[16 q, 32 keys] . V[32 keys, 16 d]           v_mfma_f32_16x16x32_bf16
// The accumulator layout of the first product (a lane holds 4 keys of one q in each of two
// tiles) is the operand layout of the second for a suitable order of the 32 keys, and values are
// cached position-contiguous ([hd][page]), so nothing passes through LDS.  The keys of a span of
// 32 are dealt to its two tiles so that those 8 keys of a lane are consecutive (tile 0 takes keys
// 0-3, 8-11, 16-19, 24-27 of the span, tile 1 the others): a lane then reads its 8 values of a
// feature with one 16-byte load.
// Each wave writes an unnormalised partial output with its maximum and sum; a second kernel
// combines the partial results of a token.
//
// Layout of an MFMA 16x16x32 operand: lane l holds, for row/column l % 16, the 8 k-values
// of group l / 16; the accumulator holds rows (l / 16) * 4 + i, column l % 16.
#include "common.h"
#include <math.h>
#include <algorithm>

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// TILES: 16-key tiles per wave (chunk = TILES * 16 keys).  Smaller chunks give more waves to
// hide latency with when the batch is small; larger ones fewer partial results.
// LOOP: a wave may take several chunks (false: exactly one, and the loop below folds away).
// BW: waves of a block.  1: the waves of a (kv head, token) are blocks of their own (blockIdx.x)
// and leave partial results for the second kernel.  More: they are the waves of one block, take
// the chunks in turn and combine their results through LDS; a single such block per (kv head,
// token) writes the output itself (with enough pairs to fill the chip that saves the second
// kernel and the trip of the partial results through memory), several of them (gridDim.x; where
// one a pair would leave compute units idle) leave one partial result each.
template <int HD, int TILES, bool LOOP, int BW>
__global__ __launch_bounds__(BW * 64) void attn_decode_split_kernel(
        const bf16_t* __restrict__ q, int q_stride,
        const bf16_t* __restrict__ kc, const bf16_t* __restrict__ vc,
        const int* __restrict__ table, int max_blocks,
        const int* __restrict__ row_of_token, const int* __restrict__ positions,
        const int* __restrict__ kv_lens, const int* __restrict__ cu_q, int H, int Hkv, int page,
        float scale, int window, int splits, float* __restrict__ part_o, float* __restrict__ part_ml,
        bf16_t* __restrict__ out, int out_stride, int rows, const int* __restrict__ single_tokens) {
    static_assert(BW == 1 || LOOP, "the waves of a block take the chunks in turn");
    extern __shared__ float lds[];                        // BW > 1: [BW][G][HD] outputs, [BW][16] maxima, [BW][16] sums
    // single_tokens (beside prompt portions): the tokens of the rows of one token, then -1; the grid
    // then spans those instead of every token of the step, most of which would have nothing to do
    const int g = blockIdx.y, t = single_tokens ? single_tokens[blockIdx.z] : (int)blockIdx.z;
    if (t < 0) return;
    // the wave's index is the same in all its lanes: said so, what depends on it alone (the chunk,
    // its pages' ids) is computed and loaded once a wave, on the scalar unit
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), col = lane & 15, grp = lane >> 4;
    const int G = H / Hkv;
    // Q^T fragments: column = query head of this group, k = head dimension
    bf16x8_t qf[HD / 32];
#pragma unroll
    for (int kk = 0; kk < HD / 32; ++kk) {
        if (col < G)
            qf[kk] = *reinterpret_cast<const bf16x8_t*>(q + (size_t)t * q_stride + (size_t)(g * G + col) * HD + kk * 32 + grp * 8);
        else
            for (int e = 0; e < 8; ++e) qf[kk][e] = (__bf16)0.f;
    }

    // Rows of one token usually come in the order of their tokens (token t is row t).  The row's
    // length and the page ids of the first chunk are asked for on that guess, together with the
    // token's row and position and before it is known whether the chunk lies within the row, so
    // that the keys can be asked for after one round trip to memory instead of three.
    constexpr int CHUNK = TILES * 16;
    const int S = BW * (int)gridDim.x;                    // waves per (kv head, token)
    int c = (int)blockIdx.x * BW + wave;
    const bool whole = BW > 1 && gridDim.x == 1;          // this block sees all the chunks and writes the output itself
    const int b_guess = min(t, rows - 1);
    int blk_of[TILES];                                    // pages of the chunk's 16-key stretches
#pragma unroll
    for (int tile = 0; tile < TILES; ++tile)
        blk_of[tile] = table[(size_t)b_guess * max_blocks + min((c * CHUNK + tile * 16) / page, max_blocks - 1)];
    int kv_len = kv_lens[b_guess];
    const int p = positions[t];
    const int b = row_of_token[t];
    if (b >= 0 && cu_q && cu_q[b + 1] - cu_q[b] != 1) return;      // rows of several tokens belong to the tiled kernel
    if (b < 0) {                                          // a padding token
        if (whole) {
            bf16_t* o_row = out + (size_t)t * out_stride + (size_t)g * G * HD;
            for (int e = threadIdx.x; e < G * HD; e += BW * 64) o_row[e] = 0;
        }
        return;
    }
    if (b != b_guess) {                                   // the guess was wrong: ask again
#pragma unroll
        for (int tile = 0; tile < TILES; ++tile)
            blk_of[tile] = table[(size_t)b * max_blocks + min((c * CHUNK + tile * 16) / page, max_blocks - 1)];
        kv_len = kv_lens[b];
    }
    const int visible = min(kv_len, p + 1);
    const int j0 = window > 0 ? max(0, p + 1 - window) : 0;
    if (visible <= j0) {                                  // nothing to see (the same for the whole block)
        if (whole) {
            bf16_t* o_row = out + (size_t)t * out_stride + (size_t)g * G * HD;
            for (int e = threadIdx.x; e < G * HD; e += BW * 64) o_row[e] = 0;
        }
        return;
    }
    const int c_last = (visible - 1) / CHUNK;
    // the combine reads the slots of the blocks whose first chunk exists: [0, min(blocks, c_last / BW + 1))
    if (!whole && (int)blockIdx.x * BW > c_last) return;

    // A wave takes the chunks c, c + S, c + 2S, ... of its row and keeps a running maximum, sum
    // and output over them, so that a long context leaves S partial results, not one per chunk.
    f32x4_t o[HD / 16];
#pragma unroll
    for (int db = 0; db < HD / 16; ++db) o[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    for (bool first = true; (LOOP || first) && c <= c_last; c += S, first = false) {
        const int c_lo = c * CHUNK;
        if (LOOP && !first) {
#pragma unroll
            for (int tile = 0; tile < TILES; ++tile)
                blk_of[tile] = table[(size_t)b * max_blocks + min((c_lo + tile * 16) / page, max_blocks - 1)];
        }
        if (c_lo + CHUNK <= j0) continue;                 // the window has passed this chunk

        // All key and value fragments of the chunk are requested before anything is computed, so
        // a wave waits for memory once a chunk.
        // Span sp = keys c_lo + 32 sp .. + 31; its tile e holds, in row r, key 8 (r / 4) + 4 e + r % 4.
        bf16x8_t kf[TILES][HD / 32];
        bf16x8_t vf[TILES / 2][HD / 16];
        bool live[TILES / 2];
#pragma unroll
        for (int sp = 0; sp < TILES / 2; ++sp) {
            const int span0 = c_lo + sp * 32;
            live[sp] = span0 < visible && span0 + 32 > j0;
            // keys: this lane's row of either tile lies in the first 16 keys of the span (col < 8) or the second
            const int kblk = live[sp] ? (col < 8 ? blk_of[2 * sp] : blk_of[2 * sp + 1]) : -1;
            const int krow = span0 + (col >> 2) * 8 + (col & 3);                  // tile 0; tile 1: + 4
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                if (kblk >= 0 && krow + 4 * e < visible) {
                    const bf16_t* kt = kc + ((size_t)kblk * Hkv + g) * (size_t)page * HD + (size_t)((krow + 4 * e) % page) * HD + grp * 8;
#pragma unroll
                    for (int kk = 0; kk < HD / 32; ++kk) kf[2 * sp + e][kk] = ld_stream16<bf16x8_t>(kt + kk * 32);
                } else {                                  // a page the window has passed, or a key not written yet
#pragma unroll
                    for (int kk = 0; kk < HD / 32; ++kk) for (int x = 0; x < 8; ++x) kf[2 * sp + e][kk][x] = (__bf16)0.f;
                }
            }
            // values: this lane's 8 keys are span0 + 8 grp .. + 7, one 16-byte piece of a feature's row
            const int vblk = live[sp] ? (grp < 2 ? blk_of[2 * sp] : blk_of[2 * sp + 1]) : -1;
            const int vkey = span0 + grp * 8;
            if (vblk >= 0 && vkey < visible) {
                const bf16_t* vt = vc + ((size_t)vblk * Hkv + g) * (size_t)page * HD + (size_t)col * page + vkey % page;
#pragma unroll
                for (int db = 0; db < HD / 16; ++db) vf[sp][db] = ld_stream16<bf16x8_t>(vt + (size_t)db * 16 * page);
                // positions never written (the rest of the last page) may hold anything, NaN included
                if (vkey + 8 > visible) {
                    const int n = visible - vkey;
#pragma unroll
                    for (int db = 0; db < HD / 16; ++db)
#pragma unroll
                        for (int x = 0; x < 8; ++x)
                            if (x >= n) vf[sp][db][x] = (__bf16)0.f;
                }
            } else {
#pragma unroll
                for (int db = 0; db < HD / 16; ++db) for (int x = 0; x < 8; ++x) vf[sp][db][x] = (__bf16)0.f;
            }
        }
        // scores: st[tile][i] = S^T[key = c_lo + 32 (tile / 2) + 8 grp + 4 (tile % 2) + i][q = col]
        f32x4_t st[TILES];
#pragma unroll
        for (int tile = 0; tile < TILES; ++tile) {
            st[tile] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kk = 0; kk < HD / 32; ++kk)
                st[tile] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[tile][kk], qf[kk], st[tile], 0, 0, 0);
        }
        // mask, scale, maximum over the keys of each q (this chunk and those before)
        float m = m_run;
#pragma unroll
        for (int tile = 0; tile < TILES; ++tile) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = c_lo + (tile >> 1) * 32 + grp * 8 + (tile & 1) * 4 + i;
                const float sc = (key < visible && key >= j0) ? st[tile][i] * scale : -INFINITY;
                st[tile][i] = sc;
                m = fmaxf(m, sc);
            }
        }
        m = fmaxf(m, __shfl_xor(m, 16, 64));
        m = fmaxf(m, __shfl_xor(m, 32, 64));
        float lsum = 0.f;
#pragma unroll
        for (int tile = 0; tile < TILES; ++tile) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float e = __expf(st[tile][i] - m);        // exp(-inf) = 0 for masked keys
                st[tile][i] = e;
                lsum += e;
            }
        }
        lsum += __shfl_xor(lsum, 16, 64);
        lsum += __shfl_xor(lsum, 32, 64);
        if (LOOP && !first) {
            // what the earlier chunks left is brought to the new maximum; m and l belong to the
            // query in this lane's column, the output rows to the queries grp*4 + i
            const float alpha = __expf(m_run - m);              // 0 if nothing was seen so far
            l_run *= alpha;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float ai = __shfl(alpha, grp * 4 + i, 64);
#pragma unroll
                for (int db = 0; db < HD / 16; ++db) o[db][i] *= ai;
            }
        }
        l_run += lsum;
        m_run = m;

        // O[q, d] += P . V over the spans: this lane's 8 keys are span keys 8 grp .. + 7, for P
        // (4 from either tile) and for V alike
#pragma unroll
        for (int sp = 0; sp < TILES / 2; ++sp) {
            if (!live[sp]) continue;
            bf16x8_t pf;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                pf[i] = (__bf16)st[2 * sp][i];
                pf[4 + i] = (__bf16)st[2 * sp + 1][i];
            }
#pragma unroll
            for (int db = 0; db < HD / 16; ++db)
                o[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf, vf[sp][db], o[db], 0, 0, 0);
        }
    }
    if constexpr (BW > 1) {
        // the waves' results meet in LDS; then every thread finishes a few outputs
        float* so = lds;                                   // [BW][G][HD]
        float* sm = lds + (size_t)BW * G * HD;              // [BW][16]
        float* sl = sm + BW * 16;                          // [BW][16]
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int qi = grp * 4 + i;
            if (qi < G) {
#pragma unroll
                for (int db = 0; db < HD / 16; ++db) so[((size_t)wave * G + qi) * HD + db * 16 + col] = o[db][i];
            }
        }
        if (grp == 0) { sm[wave * 16 + col] = m_run; sl[wave * 16 + col] = l_run; }
        __syncthreads();
        bf16_t* o_row = out + (size_t)t * out_stride + (size_t)g * G * HD;
        for (int e = threadIdx.x; e < G * HD; e += BW * 64) {
            const int qi = e / HD, d = e - qi * HD;
            float m = -INFINITY;
#pragma unroll
            for (int w = 0; w < BW; ++w) m = fmaxf(m, sm[w * 16 + qi]);
            float acc = 0.f, l = 0.f;
#pragma unroll
            for (int w = 0; w < BW; ++w) {
                // 0 for a wave without chunks (and for all of them, if a window has passed every chunk of this block)
                const float wgt = sm[w * 16 + qi] == -INFINITY ? 0.f : __expf(sm[w * 16 + qi] - m);
                acc += wgt * so[((size_t)w * G + qi) * HD + d];
                l += wgt * sl[w * 16 + qi];
            }
            if (whole) {
                o_row[e] = f32_to_bf16(acc / l);
            } else {
                // one of several blocks of this (kv head, token): its sums go to slot blockIdx.x
                const size_t slot = ((size_t)b * H + g * G + qi) * splits + blockIdx.x;
                part_o[slot * HD + d] = acc;
                if (d == 0) { part_ml[slot * 2] = m; part_ml[slot * 2 + 1] = l; }
            }
        }
        return;
    }
    // partial results in slot blockIdx.x: o[db][i] = O[q = grp*4 + i][d = db*16 + col]
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int qi = grp * 4 + i;
        if (qi < G) {
            float* dst = part_o + (((size_t)b * H + g * G + qi) * splits + blockIdx.x) * HD;   // a row of one token: indexed by row
#pragma unroll
            for (int db = 0; db < HD / 16; ++db) dst[db * 16 + col] = o[db][i];
        }
    }
    if (grp == 0 && col < G) {
        float* dst = part_ml + (((size_t)b * H + g * G + col) * splits + blockIdx.x) * 2;
        dst[0] = m_run;
        dst[1] = l_run;
    }
}

constexpr int LIST_SPAN = 32, LIST_ROWS = 64, LIST_WAVES = 512;

// How the list below is divided: spans of keys [first, end), the waves of a list of `total` spans, the first span of wave w, the wave of
// span f, and the slots a row of at most max_kv_len keys has: one a span up to 64, else as many as it meets waves whose stretches are two spans or
// more (those between its first and its last have two of its spans or more).  Stretches of one span are for short lists: 5 rows of 20 keys 10.9 -> 7.9 us.
__host__ __device__ inline int list_spans(int first, int end) { return end > first ? (end + LIST_SPAN - 1) / LIST_SPAN - first / LIST_SPAN : 0; }
__host__ __device__ inline int list_slots(int max_kv_len) {
    const int spans = (max_kv_len + LIST_SPAN - 1) / LIST_SPAN, two = spans / 2 + 1;
    return spans <= 64 ? spans : two > 64 ? two : 64;
}
__host__ __device__ inline uint32_t list_waves(uint32_t total, uint32_t most, int max_kv_len) {
    const uint32_t useful = max_kv_len <= 64 * LIST_SPAN || total <= 64 ? total : total / 2;
    return most < useful ? most : useful;
}
__host__ __device__ inline uint32_t list_from(uint32_t w, uint32_t total, uint32_t waves) { return w * total / waves; }       // (waves total < 2^32: the host's rule)
__host__ __device__ inline uint32_t list_wave_of(uint32_t f, uint32_t total, uint32_t waves) { return ((f + 1) * waves - 1) / total; }

// The same for a test that divides a list without a GPU.
extern "C" int ri_attention_list_spans(int first, int end) { return list_spans(first, end); }
extern "C" unsigned ri_attention_list_waves(unsigned total, unsigned most, int max_kv_len) { return list_waves(total, most, max_kv_len); }
extern "C" unsigned ri_attention_list_from(unsigned w, unsigned total, unsigned waves) { return list_from(w, total, waves); }
extern "C" unsigned ri_attention_list_wave_of(unsigned f, unsigned total, unsigned waves) { return list_wave_of(f, total, waves); }
extern "C" int ri_attention_list_slots(int max_kv_len) { return list_slots(max_kv_len); }

// The rows' keys as one list.  Rows differ in length, and 2,049 keys are one span more than 32 waves of 64 keys take at once, so
// a number of blocks a row leaves units idle or a few waves with twice the others' work.  Here the spans of 32
// keys of all rows (up to 64, a lane each) are numbered one after the other, and wave w of a key/value head takes the stretch
// [w total / W, (w + 1) total / W) of them, with a running maximum and sum; where a row ends it leaves that row's partial result
// in slot w - (the first wave that has a span of the row).  count[b]: the row's slots.  A span's keys and values are asked for
// while the one before it is worked on, its pages' ids a span earlier, under no lane's condition (what lies beyond the row is
// put to zero, or its score to -inf, where it is used).  Keys from max_kv_len on are not looked at, whatever kv_lens says: slots,
// page ids and the list's numbers are bounded by it.  Two waves a unit in all: more leave more partial results for the same bytes.
// The sums are O^T[d, q] = V^T . P^T, so that a query's factors lie in the lanes that hold its sums; the weights go
// to the matrix instruction as the sum of two bfloat16, which costs a bound-by-memory kernel nothing (error of the
// output against 64 bits 2.1e-3 -> 1.7e-3, that of its own rounding).
// What bounds it: the bytes, and 8 us of launches, chains of small loads and the merge.  Head 128, page 16, with the merge, us, before (blocks a
// row) / now, and the bytes at 6.87 TB/s: 43 rows of 210..3,000 keys 54.7 / 37.2 (29.2), 20 rows of 97..1,333
// 20.2 / 14.7 (6.1), 24 rows of 1,500 41 / 29 (21.5), 8 rows of 700 13.2 / 11.2, 64 rows of 2,050 95 / 92 (78).  list_pays says where it is taken.
__global__ __launch_bounds__(64, 2) void attn_decode_list_kernel(
        const bf16_t* __restrict__ q, int q_stride, const bf16_t* __restrict__ kc, const bf16_t* __restrict__ vc,
        const int* __restrict__ table, int max_blocks, const int* __restrict__ row_of_token, const int* __restrict__ positions,
        const int* __restrict__ kv_lens, int H, int Hkv, int page, int page_shift, float scale, int window, int max_kv_len, int splits,
        float* __restrict__ part_o, float* __restrict__ part_ml, int* __restrict__ count, int tokens, int rows) {
    constexpr int HD = 128, KT = 2, SPAN = LIST_SPAN;       // 16 KiB of keys and values
    const int lane = threadIdx.x, col = lane & 15, grp = lane >> 4, g = blockIdx.y, G = H / Hkv;
    // lane i: token i, its row, keys [first, end), and the spans up to and with it
    int row = -1, first = 0, end = 0, ends = 0;
    if (lane < tokens) {
        const int guess = min(lane, rows - 1);              // rows usually come in the order of their tokens
        int len = kv_lens[guess];
        const int p = positions[lane];
        row = row_of_token[lane];
        if (row >= 0 && row != guess) len = kv_lens[row];
        if (row >= 0) {                                     // else a padding token
            end = min(min(len, p + 1), max_kv_len);
            first = window > 0 ? max(0, p + 1 - window) : 0;
        }
    }
    ends = list_spans(first, end);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int up = __shfl_up(ends, o, 64);
        if (lane >= o) ends += up;
    }
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane(ends, 63);
    if (total == 0) return;
    const uint32_t W = list_waves(total, gridDim.x, max_kv_len), w = blockIdx.x;
    if (w >= W) return;
    const int f0 = (int)list_from(w, total, W), f1 = (int)list_from(w + 1, total, W);
    struct Row { int tok, row, first, end, f0, n; };        // spans [f0, f0 + n) of the list
    auto row_of = [&](int f) {                              // the row of span f < total
        const int who = __popcll(__ballot(ends <= f));      // rows that end at or before it
        Row x;
        x.tok = who;
        x.row = __builtin_amdgcn_readlane(row, who);
        x.first = __builtin_amdgcn_readlane(first, who);
        x.end = __builtin_amdgcn_readlane(end, who);
        x.n = list_spans(x.first, x.end);
        x.f0 = __builtin_amdgcn_readlane(ends, who) - x.n;
        return x;
    };

    struct Span { bf16x8_t k[KT][HD / 32], v[KT / 2][HD / 16]; };
    struct Pages { int id[KT]; };                           // of the span's stretches of 16 keys
    bf16x8_t qf[HD / 32], q_next[HD / 32];
    auto ask_query = [&](int t, bf16x8_t (&to)[HD / 32]) {      // columns beyond the group repeat its last head; nothing is kept of them
        const bf16_t* src = q + (size_t)t * q_stride + (size_t)(g * G + min(col, G - 1)) * HD + grp * 8;
#pragma unroll
        for (int kk = 0; kk < HD / 32; ++kk) to[kk] = *reinterpret_cast<const bf16x8_t*>(src + kk * 32);
    };
    const size_t page_size = (size_t)Hkv * page * HD;
    auto pages_of = [&](const Row& r, int key0, Pages& p) {
        const int* ids = table + (size_t)r.row * max_blocks;
#pragma unroll
        for (int x = 0; x < KT; ++x) {
            const int k = min(key0 + 16 * x, r.end - 1);
            p.id[x] = ids[k >> page_shift];
        }
    };
    auto slot_of = [&](int key) { return key & (page - 1); };
    auto ask = [&](Span& s, int key0, const Pages& p) {
#pragma unroll
        for (int h = 0; h < KT / 2; ++h) {
            // keys: row r of tile e is key 8 (r / 4) + 4 e + r % 4 of the half; values: the lane's 8 keys are 8 grp .. + 7
            const int k0 = key0 + 32 * h;
            const bf16_t* k = kc + (size_t)max(col < 8 ? p.id[2 * h] : p.id[2 * h + 1], 0) * page_size + (size_t)g * page * HD
                              + slot_of(k0 + (col >> 2) * 8 + (col & 3)) * HD + grp * 8;
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
                for (int kk = 0; kk < HD / 32; ++kk) s.k[2 * h + e][kk] = ld_stream16<bf16x8_t>(k + 4 * e * HD + kk * 32);
            const bf16_t* v = vc + (size_t)max(grp < 2 ? p.id[2 * h] : p.id[2 * h + 1], 0) * page_size + (size_t)g * page * HD
                              + col * page + slot_of(k0 + grp * 8);
#pragma unroll
            for (int db = 0; db < HD / 16; ++db) s.v[h][db] = ld_stream16<bf16x8_t>(v + (size_t)db * 16 * page);
        }
    };
    f32x4_t o[HD / 16];
    float m_run = -INFINITY, l_run = 0.f;                   // l_run: this lane's keys alone, until the row's end
    auto clear = [&]() {
#pragma unroll
        for (int db = 0; db < HD / 16; ++db) o[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        m_run = -INFINITY;
        l_run = 0.f;
    };
    // keys [lo, hi) of a row are its own; p are the span's pages
    auto work = [&](Span& s, int key0, int lo, int hi, const Pages& p) {
        f32x4_t st[KT];
#pragma unroll
        for (int t = 0; t < KT; ++t) {
            st[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kk = 0; kk < HD / 32; ++kk) st[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(s.k[t][kk], qf[kk], st[t], 0, 0, 0);
        }
        const bool cut = key0 < lo || key0 + SPAN > hi;
        float m = m_run;
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = key0 + (t >> 1) * 32 + grp * 8 + (t & 1) * 4 + i;        // of query col
                float sc = st[t][i] * scale;
                if (cut) sc = key >= lo && key < hi ? sc : -INFINITY;
                st[t][i] = sc;
                m = fmaxf(m, sc);
            }
        m = fmaxf(m, __shfl_xor(m, 16, 64));
        m = fmaxf(m, __shfl_xor(m, 32, 64));
        const float top = m > -INFINITY ? m : 0.f;          // (a span whose every score is -inf has no weight, and takes none from the others)
        const float alpha = __expf(m_run - top);            // 0 if nothing was seen so far
        float sum = 0.f;
        bf16x8_t pf[KT / 2], rest[KT / 2];
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float x = __expf(st[t][i] - top);     // exp(-inf) = 0 for masked keys
                sum += x;
                const __bf16 y = (__bf16)x;
                pf[t >> 1][4 * (t & 1) + i] = y;
                rest[t >> 1][4 * (t & 1) + i] = (__bf16)(x - (float)y);
            }
        l_run = l_run * alpha + sum;
        m_run = m;
#pragma unroll
        for (int db = 0; db < HD / 16; ++db)
#pragma unroll
            for (int i = 0; i < 4; ++i) o[db][i] *= alpha;
        bool gone = false;
#pragma unroll
        for (int x = 0; x < KT; ++x) gone |= p.id[x] < 0;
        if (cut || gone) {                                  // slots never written and pages given back may hold anything, NaN included
#pragma unroll
            for (int h = 0; h < KT / 2; ++h) {
                const int there = (grp < 2 ? p.id[2 * h] : p.id[2 * h + 1]) >= 0 ? hi - (key0 + 32 * h + grp * 8) : 0;
#pragma unroll
                for (int db = 0; db < HD / 16; ++db)
#pragma unroll
                    for (int x = 0; x < 8; ++x)
                        if (x >= there) s.v[h][db][x] = (__bf16)0.f;
            }
        }
#pragma unroll
        for (int h = 0; h < KT / 2; ++h)
#pragma unroll
            for (int db = 0; db < HD / 16; ++db) {
                o[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(s.v[h][db], pf[h], o[db], 0, 0, 0);
                o[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(s.v[h][db], rest[h], o[db], 0, 0, 0);
            }
    };
    auto leave = [&](int b, int f, int n) {                 // row b: spans [f, f + n) of the list
        const uint32_t w0 = list_wave_of(f, total, W);
        float l = l_run;
        l += __shfl_xor(l, 16, 64);
        l += __shfl_xor(l, 32, 64);
        if (col < G) {
            const size_t slot = ((size_t)b * H + g * G + col) * splits + (w - w0);
#pragma unroll
            for (int db = 0; db < HD / 16; ++db)
                *reinterpret_cast<float4*>(part_o + slot * HD + db * 16 + grp * 4) = make_float4(o[db][0], o[db][1], o[db][2], o[db][3]);
            if (grp == 0) *reinterpret_cast<float2*>(part_ml + slot * 2) = make_float2(m_run, l);
        }
        if (w == w0 && g == 0 && lane == 0) count[b] = (int)(list_wave_of(f + n - 1, total, W) - w0 + 1);
    };
    clear();
    Span sa, sb;
    // the span that is worked on, and the one after it, whose pages' ids are asked for before its turn comes
    Row now = row_of(f0), next = now;
    Pages p, np;
    int key = (now.first / SPAN + f0 - now.f0) * SPAN, next_key = key;
    auto after = [&](int f, const Row& r, int at) {         // span f follows the one at key `at` of row r
        next = r;
        next_key = at + SPAN;
        if (f == r.f0 + r.n && f < f1) {
            next = row_of(f);
            next_key = next.first / SPAN * SPAN;
        }
        pages_of(next, next_key, np);
    };
    ask_query(now.tok, qf);
    pages_of(now, key, p);
    ask(sa, key, p);
    after(f0 + 1, now, key);
    // one span: the one after it is asked for first, perhaps of another row
    auto step = [&](Span& here, Span& there, int f) {
        const Row r = now;
        const Pages pages = p;
        const int at = key;
        const bool last = f + 1 == r.f0 + r.n;              // of its row
        if (last) ask_query(next.tok, q_next);
        ask(there, next_key, np);
        now = next;
        key = next_key;
        p = np;
        after(f + 2, now, key);
        work(here, at, r.first, r.end, pages);
        if (last) {
            leave(r.row, r.f0, r.n);
            clear();
#pragma unroll
            for (int kk = 0; kk < HD / 32; ++kk) qf[kk] = q_next[kk];
        }
    };
    int f = f0;
    for (; f + 2 < f1; f += 2) {
        step(sa, sb, f);
        step(sb, sa, f + 1);
    }
    if (f + 1 < f1) {
        step(sa, sb, f);
        work(sb, key, now.first, now.end, p);
    } else {
        work(sa, key, now.first, now.end, p);
    }
    leave(now.row, now.f0, now.n);
}

// One block of CW waves per (token, head).  The partial results of the chunks are rows of HD
// floats; a wave reads them 16 bytes a lane, 64 / (HD / 4) rows per load instruction, several
// instructions in flight, and each wave takes its share of the rows, so that long contexts
// (hundreds of chunks) are combined by more than a trickle of 4-byte loads.
template <int HD, int CW>
__global__ __launch_bounds__(CW * 64) void attn_decode_combine_kernel(
        const float* __restrict__ part_o, const float* __restrict__ part_ml, int splits, int chunk,
        const int* __restrict__ row_of_token, const int* __restrict__ positions,
        const int* __restrict__ kv_lens, const int* __restrict__ cu_q, int H, int window,
        bf16_t* __restrict__ out, int out_stride, int rows, const int* __restrict__ single_tokens, const int* __restrict__ count) {
    constexpr int LPP = HD / 4;               // lanes per row of partial results (a float4 each)
    constexpr int PPW = 64 / LPP;             // rows per load instruction of a wave
    constexpr int UNR = 4;                    // load instructions in flight
    __shared__ float red[16];
    __shared__ float4 accs[CW][LPP];
    __shared__ float ls[CW];
    const int t = single_tokens ? single_tokens[blockIdx.x] : (int)blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
    if (t < 0) return;
    const int lane = tid & 63, wave = tid >> 6;
    bf16_t* o = out + (size_t)t * out_stride + (size_t)h * HD;
    // as in the first kernel, the row is guessed to be the token's index, and what depends on it
    // (the row's length, this thread's first maximum) is asked for together with the row itself
    const int b_guess = min(t, rows - 1);
    int kv_len = kv_lens[b_guess];
    float m_first = tid < splits ? part_ml[(((size_t)b_guess * H + h) * splits + tid) * 2] : -INFINITY;
    const int p = positions[t];
    const int b = row_of_token[t];
    if (b >= 0 && cu_q && cu_q[b + 1] - cu_q[b] != 1) return;
    if (b >= 0 && b != b_guess) {
        kv_len = kv_lens[b];
        m_first = tid < splits ? part_ml[(((size_t)b * H + h) * splits + tid) * 2] : -INFINITY;
    }
    int visible = 0, j0 = 0;
    if (b >= 0) {
        visible = min(kv_len, p + 1);
        if (count) visible = min(visible, chunk);        // (of the list's form: the longest length, which its spans end at)
        j0 = window > 0 ? max(0, p + 1 - window) : 0;
    }
    if (visible <= j0) {                      // a padding token, or nothing to see: zeros
        for (int e = tid; e < HD; e += CW * 64) o[e] = 0;
        return;
    }
    // the waves of the first kernel left one slot each; those beyond the row's last chunk none
    const int n = count ? count[b] : min(splits, (visible - 1) / chunk + 1);
    const float2* ml = reinterpret_cast<const float2*>(part_ml) + ((size_t)b * H + h) * splits;
    const float4* po = reinterpret_cast<const float4*>(part_o + ((size_t)b * H + h) * splits * HD);
    float m = tid < n ? m_first : -INFINITY;             // slots beyond n hold nothing of this step
    for (int i = tid + CW * 64; i < n; i += CW * 64) m = fmaxf(m, ml[i].x);
    m = CW > 1 ? block_max(m, red) : wave_max(m);
    const int sub = lane / LPP, colv = lane % LPP;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    float l = 0.f;
    for (int i0 = wave * PPW + sub; i0 < n; i0 += CW * PPW * UNR) {
        float4 pv[UNR];
        float2 mv[UNR];
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const int i = i0 + u * CW * PPW;
            const bool ok = i < n;
            pv[u] = ok ? po[(size_t)i * LPP + colv] : make_float4(0.f, 0.f, 0.f, 0.f);
            mv[u] = ok ? ml[i] : make_float2(-INFINITY, 0.f);
        }
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const float wgt = __expf(mv[u].x - m);                // 0 for rows beyond the end
            acc.x += wgt * pv[u].x; acc.y += wgt * pv[u].y; acc.z += wgt * pv[u].z; acc.w += wgt * pv[u].w;
            if (colv == 0) l += wgt * mv[u].y;
        }
    }
    // rows that share a wave, then the waves
#pragma unroll
    for (int off = LPP; off < 64; off <<= 1) {
        acc.x += __shfl_xor(acc.x, off, 64); acc.y += __shfl_xor(acc.y, off, 64);
        acc.z += __shfl_xor(acc.z, off, 64); acc.w += __shfl_xor(acc.w, off, 64);
    }
    l = wave_sum(l);
    if (CW > 1) {
        if (lane < LPP) accs[wave][lane] = acc;
        if (lane == 0) ls[wave] = l;
        __syncthreads();
        if (wave > 0) return;
        for (int w = 1; w < CW; ++w) {
            if (lane < LPP) { const float4 a = accs[w][lane]; acc.x += a.x; acc.y += a.y; acc.z += a.z; acc.w += a.w; }
            l += ls[w];
        }
    }
    if (lane < LPP) {
        const float inv = 1.f / l;
        uint2 r;
        r.x = (uint32_t)f32_to_bf16(acc.x * inv) | ((uint32_t)f32_to_bf16(acc.y * inv) << 16);
        r.y = (uint32_t)f32_to_bf16(acc.z * inv) | ((uint32_t)f32_to_bf16(acc.w * inv) << 16);
        *reinterpret_cast<uint2*>(o + lane * 4) = r;
    }
}

// keys per wave: 128 when there are waves enough anyway, else 64 (with 8 or fewer rows of 2,000
// keys, chunks of 32, 64 and 128 keys take the same time within 1 %: the kernel is not bound by
// the number of its waves or of its load instructions)
static int decode_chunk(int T, int Hkv, int hd, int max_kv_len) {
    if (hd == 128) return 64;
    const long long waves128 = (long long)T * Hkv * ((max_kv_len + 127) / 128);
    return waves128 >= 4096 ? 128 : 64;
}

extern "C" size_t ri_attention_decode_workspace(int rows, int H, int hd, int max_kv_len) {
    const int blocks = (max_kv_len + 63) / 64;                  // no form of blocks a row leaves more; the list is head 128's
    const size_t splits = (size_t)(hd == 128 ? std::max(list_slots(max_kv_len), blocks) : blocks);
    return ((size_t)rows * H * splits * (hd + 2) + rows) * sizeof(float);
}

extern "C" int ri_attention_decode_supported(int H, int Hkv, int hd, int page) {
    return (hd == 64 || hd == 128) && page % 16 == 0 && Hkv > 0 && H % Hkv == 0 && H / Hkv <= 16;
}

// Whether a step of T single tokens alone takes the list of spans.  It divides rows of any lengths evenly, and pays a merge for it.  Blocks a row are better
// where one block a (key/value head, token) pair nearly fills the chip and writes its output itself, for rows that are short or alike.  Which rows are is not
// known here, only the longest length the step was planned for, so 129 to 256 pairs keep their blocks up to 1,024 keys.
// Measured, us, head 128, blocks a row / list, 8 heads: 24 equal rows of 20 keys 5.5 / 8.2, of 100 6.5 / 9.2, of 700 16.6 / 18.5, of 1,500 32.6 / 27.6, ragged ones
// up to 1,000 20.3 / 13.7 (given up for the equal ones), up to 3,000 42 / 24; 32 rows, equal 700 18.5 / 21.1, 1,500 35.5 / 36.4, 2,050 46.6 / 48.3, 4,000 86 / 84,
// ragged up to 3,000 54 / 28 (kept).  Elsewhere: 8 rows of 20 9.0 / 7.8, of 2,050 18.4 / 17.9, 12 of 100 9.4 / 8.6, 40 of 100 18 / 10, 64 of 100 11.8 / 12.0, of 700
// 35 / 34, ragged up to 1,000 34 / 21; the worst, 56 of 65 10.2 / 11.3.  Fewer than 12 pairs: 3 ragged rows of 2 heads up to 3,000 10.5 / 11.2.  Head 64:
// 43 rows of 210..3,000 37 / 25, but 16 rows of 2,050 18.4 / 19.8 and 32 27 / 31: never.
static bool list_pays(long long pairs, int hd, int max_kv_len) {
    return hd == 128 && pairs >= 12 && !(pairs > 128 && pairs <= 256 && max_kv_len <= 1024);
}

// Whether a step of T single tokens alone goes as a list: what it takes (rows for the lanes of a wave, w total below 2^32), and where it pays.
// (No more rows than lanes: a first form that read more than 64 rows in groups faulted the GPU once, with 100 rows of 700 keys.  The cause was not shown, that
// form is not in the code, and such steps take blocks a row; whoever lifts the limit has that to explain first.)
extern "C" int ri_attention_decode_as_list(int T, int Hkv, int hd, int page, int max_kv_len) {
    const long long spans = (long long)T * ((max_kv_len + LIST_SPAN - 1) / LIST_SPAN + 1);
    return T >= 3 && T <= LIST_ROWS && (page & (page - 1)) == 0 && spans < (1ll << 32) / LIST_WAVES && list_pays((long long)T * Hkv, hd, max_kv_len);
}

extern "C" int ri_attention_decode(
        const void* q, int q_stride, void* out, int out_stride,
        const void* kc, const void* vc, int num_pages, int page, int H, int Hkv, int hd,
        const int* table, int max_blocks, const int* row_of_token, const int* positions,
        const int* kv_lens, const int* cu_q, int T, int rows, int max_kv_len, float scale, int window,
        void* workspace, size_t workspace_bytes, int singles, const int* single_tokens, int pair_blocks,
        hipStream_t stream) {
    // singles: how many of the T tokens are rows of one token, at most (the others belong to longer
    // portions and are left alone); <= 0: all of them.  It steers how the work is divided, and with
    // single_tokens (their `singles` flat token indices, -1 where there are fewer; may be null) the
    // grids span those tokens only: a step of a 256-token portion beside 8 single tokens otherwise
    // starts 8,448 blocks for the 256 that have work, 42 us instead of 16.
    RI_REQUIRE(ri_attention_decode_supported(H, Hkv, hd, page),
               "ri_attention_decode: needs head size 64 or 128, pages that are multiples of 16 and at most 16 "
               "query heads per kv head; got hd=%d page=%d H=%d Hkv=%d", hd, page, H, Hkv);
    RI_REQUIRE(T >= 0 && max_kv_len > 0 && max_blocks > 0 && num_pages > 0 && window >= 0, "ri_attention_decode: bad sizes");
    RI_REQUIRE(q_stride >= H * hd && out_stride >= H * hd && q_stride % 8 == 0 && out_stride % 4 == 0, "ri_attention_decode: bad row strides");
    RI_REQUIRE((long long)max_blocks * page >= max_kv_len, "ri_attention_decode: block table shorter than max_kv_len");
    if (T == 0) return 0;
    RI_REQUIRE(T <= 65535 && Hkv <= 65535, "ri_attention_decode: grid too large");
    RI_REQUIRE(q && out && kc && vc && table && row_of_token && positions && kv_lens && workspace, "ri_attention_decode: null pointer");
    RI_REQUIRE((uintptr_t)q % 16 == 0 && (uintptr_t)kc % 16 == 0 && (uintptr_t)vc % 16 == 0 && (uintptr_t)out % 8 == 0 && (uintptr_t)workspace % 16 == 0,
               "ri_attention_decode: operands must be 16-byte aligned (the output 8-byte)");
    RI_REQUIRE(rows >= 1, "ri_attention_decode: %d tokens but no rows", T);
    RI_REQUIRE(workspace_bytes >= ri_attention_decode_workspace(rows, H, hd, max_kv_len), "ri_attention_decode: workspace too small");
    const int busy = singles > 0 && singles < T ? singles : T;      // tokens that have work
    const int chunk = decode_chunk(busy, Hkv, hd, max_kv_len);
    // One wave per chunk while that keeps the number of waves and of partial results moderate;
    // beyond, about 2048 waves (two per SIMD) take several chunks each, the same number as
    // nearly as it divides, which bounds what the second kernel has to read.
    const int nchunks = (max_kv_len + chunk - 1) / chunk;
    const long long rows_heads = (long long)busy * Hkv;
    int splits = nchunks;
    if (nchunks > 64 || nchunks * rows_heads > 16384) {
        const long long cap = 2048 / rows_heads > 1 ? 2048 / rows_heads : 1;
        if (nchunks > cap) {
            const int per = (int)((nchunks + cap - 1) / cap);
            splits = (nchunks + per - 1) / per;
        }
    }
    // Blocks of several waves (as many as their registers allow) that take a pair's chunks in turn
    // and combine through LDS: one block a (kv head, token) pair that writes the output itself, or
    // several that leave a partial result each.  A compute unit holds one such block, and the time
    // is that of the fullest unit: the number of blocks a pair is the one (up to 8, and no more
    // than give every wave a chunk of the longest row) that fills whole rounds of the chip's 256
    // units best, where one a pair would leave a fifth of them idle or more; if that makes blocks
    // enough and leaves a wave at most 8 chunks (with 512 pairs or more any number); else the form
    // of one wave a chunk above.  Measured against what
    // ran before, head 128, us: 8 rows of 2,048 keys 20.3 -> 17.9 (4 blocks a pair), 16 rows
    // 43.1 -> 28.7 (2), 24 rows 45.9 -> 43.5 (4); 4,096 keys: 8 rows 34.6 -> 28.4, 16 rows 79.0 ->
    // 50.6, 4 rows 20.3 -> 18.0 (8); head 64: 16 rows of 2,048 keys 23.8 -> 18.1, 8 rows of 4,096
    // 20.7 -> 18.1.  pair_blocks: 0 lets the entry point choose, 1 forbids several blocks a pair,
    // more asks for that many.
    if (pair_blocks == 0 && !cu_q && ri_attention_decode_as_list(T, Hkv, hd, page, max_kv_len)) {
        const long long spans = (long long)T * ((max_kv_len + LIST_SPAN - 1) / LIST_SPAN + 1);
        const int W = (int)std::max(1ll, std::min<long long>(LIST_WAVES / Hkv, spans));
        const int slots = list_slots(max_kv_len);
        float* sums = (float*)workspace;
        float* ml = sums + (size_t)rows * H * slots * hd;
        int* count = (int*)(ml + (size_t)rows * H * slots * 2);
        attn_decode_list_kernel<<<dim3(W, Hkv), 64, 0, stream>>>(
            (const bf16_t*)q, q_stride, (const bf16_t*)kc, (const bf16_t*)vc, table, max_blocks, row_of_token, positions, kv_lens, H, Hkv,
            page, __builtin_ctz((unsigned)page), scale, window, max_kv_len, slots, sums, ml, count, T, rows);
        RI_LAUNCHED("ri_attention_decode(list)");
        // a row has as many slots as waves, at most
        const bool one = std::min(slots, W) <= 64;
        auto combine = one ? attn_decode_combine_kernel<128, 1> : attn_decode_combine_kernel<128, 4>;
        combine<<<dim3(T, H), one ? 64 : 256, 0, stream>>>(sums, ml, slots, max_kv_len, row_of_token, positions, kv_lens, nullptr, H, window, (bf16_t*)out,
                                                           out_stride, rows, nullptr, count);
        RI_LAUNCHED("ri_attention_decode(combine)");
        return 0;
    }
    const int bw_ = hd == 64 ? 16 : 8;
    const int chunks64_ = (max_kv_len + 63) / 64;
    const bool lds_ok = (size_t)bw_ * ((size_t)(H / Hkv) * hd + 32) * sizeof(float) <= 64 * 1024;
    int nblk = 0;                                         // 0: one wave a chunk; 1: one block a pair; more: several
    if (pair_blocks > 1) {
        nblk = std::min(pair_blocks, std::max(chunks64_ / bw_, 1));
    } else if (lds_ok && rows_heads >= 32) {
        const int max_n = pair_blocks == 1 ? 1 : std::max(std::min(chunks64_ / bw_, 8), 1);
        auto fill = [&](int n) {
            const long long blocks = rows_heads * n;
            return (double)blocks / (256.0 * (double)((blocks + 255) / 256));
        };
        nblk = 1;
        if (fill(1) < 0.8) {                              // else one block a pair wastes little (56 rows: four a pair lose 10-25 %)
            double best = 0.0;
            for (int n = 1; n <= max_n; ++n)
                if (fill(n) > best + 1e-9) { best = fill(n); nblk = n; }
        }
        const bool few_chunks_a_wave = chunks64_ <= bw_ * 8 * nblk || rows_heads >= 512;
        // Blocks enough: 128 of one a pair (measured with caches larger than the last-level cache:
        // from 128 pairs on 6 % faster than one wave a chunk, 20 % at 256; at 96 pairs 10 % slower);
        // of several a pair 192, and 256 at head 64, where a block of 16 waves costs more to start
        // and to combine (8 rows of 3,072 keys: 3 blocks a pair lose 4 %)
        const long long min_blocks = nblk == 1 ? 128 : (hd == 64 ? 256 : 192);
        if (rows_heads * nblk < min_blocks || !few_chunks_a_wave) nblk = 0;
    }
    RI_REQUIRE(nblk == 0 || lds_ok, "ri_attention_decode: %d heads a kv head are too many for blocks of several waves", H / Hkv);
    if (nblk > 1) splits = nblk;
    const int* sel = (single_tokens && singles > 0 && singles < T) ? single_tokens : nullptr;
    const int TZ = sel ? singles : T;                     // tokens the grids span
    float* part_o = (float*)workspace;
    float* part_ml = part_o + (size_t)rows * H * splits * hd;
#define RI_DECODE_ARGS (const bf16_t*)q, q_stride, (const bf16_t*)kc, (const bf16_t*)vc, table, max_blocks, row_of_token, positions, kv_lens, cu_q, H, Hkv, page, scale, window, splits, part_o, part_ml, (bf16_t*)out, out_stride, rows, sel
    if (nblk > 0) {
        const int G = H / Hkv;
        const size_t lds_bytes = (size_t)bw_ * ((size_t)G * hd + 32) * sizeof(float);
        dim3 gridh(nblk, Hkv, TZ);
        if (hd == 64) attn_decode_split_kernel<64, 4, true, 16><<<gridh, 16 * 64, lds_bytes, stream>>>(RI_DECODE_ARGS);
        else attn_decode_split_kernel<128, 4, true, 8><<<gridh, 8 * 64, lds_bytes, stream>>>(RI_DECODE_ARGS);
        RI_LAUNCHED("ri_attention_decode(blocks)");
        if (nblk == 1) return 0;                          // the block has written the output itself
        dim3 grid2(TZ, H);
        const int block_keys = 64 * bw_;                  // a block's first chunk begins a multiple of this many keys in
        if (hd == 64) attn_decode_combine_kernel<64, 1><<<grid2, 64, 0, stream>>>(part_o, part_ml, splits, block_keys, row_of_token, positions, kv_lens, cu_q, H, window, (bf16_t*)out, out_stride, rows, sel, nullptr);
        else attn_decode_combine_kernel<128, 1><<<grid2, 64, 0, stream>>>(part_o, part_ml, splits, block_keys, row_of_token, positions, kv_lens, cu_q, H, window, (bf16_t*)out, out_stride, rows, sel, nullptr);
        RI_LAUNCHED("ri_attention_decode(combine)");
        return 0;
    }
    dim3 grid(splits, Hkv, TZ);
    dim3 grid2(TZ, H);
    const bool loop = splits < nchunks;
#define RI_DECODE_LAUNCH(HD_, TILES_) do { \
        if (loop) attn_decode_split_kernel<HD_, TILES_, true, 1><<<grid, 64, 0, stream>>>(RI_DECODE_ARGS); \
        else attn_decode_split_kernel<HD_, TILES_, false, 1><<<grid, 64, 0, stream>>>(RI_DECODE_ARGS); } while (0)
    if (hd == 64 && chunk == 128) RI_DECODE_LAUNCH(64, 8);
    else if (hd == 64) RI_DECODE_LAUNCH(64, 4);
    else RI_DECODE_LAUNCH(128, 4);
#undef RI_DECODE_LAUNCH
#undef RI_DECODE_ARGS
    RI_LAUNCHED("ri_attention_decode");
    // more waves per (token, head) where there are many chunks to combine
#define RI_COMBINE_ARGS part_o, part_ml, splits, chunk, row_of_token, positions, kv_lens, cu_q, H, window, (bf16_t*)out, out_stride, rows, sel, nullptr
    if (hd == 64 && splits <= 64) attn_decode_combine_kernel<64, 1><<<grid2, 64, 0, stream>>>(RI_COMBINE_ARGS);
    else if (hd == 64) attn_decode_combine_kernel<64, 4><<<grid2, 256, 0, stream>>>(RI_COMBINE_ARGS);
    else if (splits <= 32) attn_decode_combine_kernel<128, 1><<<grid2, 64, 0, stream>>>(RI_COMBINE_ARGS);
    else attn_decode_combine_kernel<128, 4><<<grid2, 256, 0, stream>>>(RI_COMBINE_ARGS);
#undef RI_COMBINE_ARGS
    RI_LAUNCHED("ri_attention_decode(combine)");
    return 0;
}
