// The state walk of recurrent.hip for prompts, 32 tokens at a time on the matrix instructions:
//
//   delta form:  S_t = diag(w_t) S_(t-1) - b_t (u_t^T S_(t-1)) + k_t v_t^T,   o_t = S_t^T r_t
//   decay form:  S_t = d S_(t-1) + k_t v_t^T,                                 o_t = S_t^T r_t
//
// per head, S of [dk][dv], b = a * u.  Token by token that is a chain of thousands of short steps on a quarter of
// the chip's SIMDs.  Within a chunk of C tokens, with W_t = w_1 * .. * w_t (per key channel) and
//   U_t = u_t W_(t-1),   R_t = r_t W_t,   K_t = k_t / W_t,   B_t = b_t / W_t,   K~ = K W_C,   B~ = B W_C,
// the tokens' d_t = u_t^T S_(t-1) solve (I + L) D = U S_0 + N V with L, N the strictly lower parts of U B^T and U K^T.
// With T = (I + L)^-1, the lower parts A_k, A_b of R K^T, R B^T, and P = A_b T, G = B~^T T (dk x C),
//   o   = (R - P U) S_0 + (A_k - P N) V,
//   S_C = (diag(W_C) - G U) S_0 + (K~^T - G N) V.
// Everything but S_0 is the chunk's own: `chunk_operators_kernel` makes it for all chunks at once (a block a
// chunk and head), and `chunk_states_kernel` passes the state through the chunks: one product of dk x dk and one of
// C x dk against 16 of its columns a block.  The decay form has powers of d in place of the operators.
//
// W only ever divides what is multiplied by a later W: a ratio W_t / W_s is as exact as the product of the decays
// between, however small both are.  That needs W_C > 0: the caller takes this form where the design bounds the
// decays (w >= exp(-decay_c)).  A substitution and not a product of powers of L: where keys repeat, those grow
// beyond what cancels.
//
// The walk rounds a state once a token, in every element; a chunk has several products between two roundings of the
// state, and where keys share a direction those cancel.  With sums in 32 bits its states were up to 2.4 times further
// from 64-bit arithmetic than the walk's.  So all that a chunk computes from its scaled vectors (32 bits each) is 64-bit,
// on v_mfma_f64_16x16x4_f64, rounded where it is stored for the states; M is stored without W_C, so that what is rounded
// is only what the chunk changes; and the new state is rounded once.  Errors against 64 bits, of the walk's, outputs / states,
// rows of 32 to 300 tokens: random keys 0.65 / 0.90, keys around one direction 0.83 / 0.87, one repeated key 0.98 / 0.99, decay
// form 0.69 to 0.76 / 0.34 to 0.39.  (A decay as fast as 0.5 a token behind a chunk that is not whole: states up to 1.2 of
// half a unit in the last place, outputs 0.4.)
//
// What holds the tokens of a chunk apart is zeros, which a value that is not finite passes.  A chunk and head whose operators
// are not finite (a token's vectors were not, or k / W_t left the range of 32 bits) is therefore only marked; the states
// stop in front of it, and the walk does that head of that row from there on, so that every token gets what the walk gives.
//
// 2,048 tokens of 32 heads of 64, us a layer, the walk / this: delta form 1174 / 223, decay form 789 / 96; 24 heads of 128: 1692 / 583, 977 /
// 182.  The operators (163 and 50 of the first two) are bound by the steps of a block following each other (two
// blocks a compute unit), the states (86, 55) by the chain of chunks: 64 chunks of about 1.3 us, 0.5 of which are its matrix instructions
// (101, 69 with two waves, and with loads under a lane's condition, which the compiled loop waited for, 123 and 69).
#include "common.h"
#include <mutex>

namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef double f64x4_t __attribute__((ext_vector_type(4)));

constexpr int C = 32;                   // tokens a chunk

struct ChunkArgs {
    const bf16_t *r, *k, *v, *wl, *al;
    int r_stride, k_stride, v_stride, wl_stride, al_stride;
    const float *w0, *ab, *decay;
    float* state;
    float* out;
    int out_stride;
    const int *cu_q, *q_start, *slots;
    int H, silu_in, min_tokens;
    float unit_eps, decay_c;
    const float *rot_cos, *rot_sin;
    int rot;
    float k_scale;
    const int* rows;                    // the grid's rows, then -1 (null: all, in order)
    float* ws;                          // [row of the grid][chunk of the segment][head][Unit::SIZE]
    int* from;                          // [row][head][dv / 16]: the token that the walk goes on from
    int c0, seg;                        // the segment's first chunk of every row, its chunks
};

__device__ __forceinline__ float sigmoid_(float z) { return __fdividef(1.f, 1.f + __expf(-z)); }
__device__ __forceinline__ float silu_(float z) { return __fdividef(z, 1.f + __expf(-z)); }

// Floats of a chunk and head in the workspace: R' [2 tiles of 16 tokens][dk / 16][64][4], S_add [dv / 16][dk / 16][64][4]
// and, in the delta form, M [dk / 16][dk / 16][64][4] without its diagonal part, W_C [dk]: each in the order the lanes of
// chunk_states_kernel read it; BAD: not zero where something in it is not finite.
template <int DK, int DV, bool DELTA>
struct Unit {
    static constexpr int R = 0, S = C * DK, M = S + DK * DV, W = M + (DELTA ? DK * DK : 0), BAD = W + (DELTA ? DK : 0), SIZE = BAD + 4;
};
__device__ __forceinline__ bool endless(float x) { return !(fabsf(x) < __builtin_inff()); }

// d to the power n (0 <= n <= C)
__device__ __forceinline__ double power(float d, int n) {
    double p = 1.0, q = (double)d;
    for (int m = n; m > 0; m >>= 1) {
        if (m & 1) p *= q;
        q *= q;
    }
    return p;
}

// acc += A B over the tokens 4 S0 .. 4 S1 of a chunk, in 64 bits (v_mfma_f64_16x16x4_f64): lane 16 g + i brings row or column i
// and token 4 s + g, and has results (4 e + g, i) in element e.  Fed with row turned(i) in the place of i, it has rows
// 4 g + e: four consecutive ones.
template <int S0, int S1, typename FA, typename FB>
__device__ __forceinline__ f64x4_t product(f64x4_t acc, int g, FA a, FB b) {
#pragma unroll
    for (int s = S0; s < S1; ++s) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a(4 * s + g), b(4 * s + g), acc, 0, 0, 0);
    return acc;
}
__device__ __forceinline__ int turned(int i) { return 4 * (i & 3) + (i >> 2); }

// Two lower triangles of C x C share one array of C x (C + 1): (t, s) of the first is at t (C + 1) + s, of the second at
// s (C + 1) + t + 1.
constexpr int TP = C + 1;
__device__ __forceinline__ double first_of(const double* m, int t, int s) { const double x = m[t * TP + s]; return s <= t ? x : 0.0; }
__device__ __forceinline__ double second_of(const double* m, int t, int s) { const double x = m[s * TP + t + 1]; return s <= t ? x : 0.0; }
__device__ __forceinline__ double second_strictly(const double* m, int t, int s) { const double x = m[s * TP + t + 1]; return s < t ? x : 0.0; }

// LDS of a block, in floats
template <int DK, int DV, bool DELTA>
struct Lds {
    static constexpr int KP = DK + 4, VP = DV + 4, HP = DK + 2;
    static constexpr int R = 0, U = R + C * KP, V = U + (DELTA ? C * KP : 0), K = V + C * VP, B = K + C * KP,
                         G = B + (DELTA ? C * KP : 0), A = G + (DELTA ? 2 * C * HP : 0), T = A + 2 * C * TP,
                         W = T + (DELTA ? 2 * C * TP : 0), SIZE = W + 2 * (DELTA ? DK : C + 1);
    static_assert(G % 2 == 0 && A % 2 == 0 && T % 2 == 0 && W % 2 == 0, "64-bit numbers lie at even places");
};

template <int DK, int DV, bool DELTA>
__global__ __launch_bounds__(256) void chunk_operators_kernel(const ChunkArgs a) {
    using At = Lds<DK, DV, DELTA>;
    constexpr int KP = At::KP, VP = At::VP, HP = At::HP;
    constexpr int EK = DK / 64 > 0 ? DK / 64 : 1, TK = DK / 32, TV = DV / 32;
    using U = Unit<DK, DV, DELTA>;
    const int b = a.rows ? a.rows[blockIdx.z] : (int)blockIdx.z, h = blockIdx.y, cs = blockIdx.x, c = a.c0 + cs;
    if (b < 0) return;
    const int t_lo = a.cu_q[b], n = a.cu_q[b + 1] - t_lo;
    if (n < a.min_tokens || c * C >= n) return;
    const int nc = min(C, n - c * C), t0 = t_lo + c * C;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i16 = lane & 15, g = lane >> 4;
    extern __shared__ __align__(16) float lds[];
    float* Rm = lds + At::R;                  // [C][KP]: r, then R
    float* Um = lds + At::U;                  // delta: u, then U
    float* Vm = lds + At::V;                  // [C][VP]
    float* Km = lds + At::K;                  // k, then K
    float* Bm = lds + At::B;                  // delta: b, then B
    float* Ws = lds + At::G;                  // delta: [C][DK] of w, until W is made
    double* Gs = reinterpret_cast<double*>(lds + At::G);       // delta: [C][HP] of G
    double* Hs = reinterpret_cast<double*>(lds + At::K);       // delta: [C][HP] of H, in the place of K and B
    double* A2 = reinterpret_cast<double*>(lds + At::A);       // A_k, then E; delta: and A_b, then P
    double* T2 = reinterpret_cast<double*>(lds + At::T);       // delta: L, then T; and N
    double* Wc = reinterpret_cast<double*>(lds + At::W);       // delta: [DK] of W_C; else powers of d, 0 .. C
    static_assert(2 * HP <= 2 * KP, "H fits where K and B were");
    float* unit = a.ws + (((size_t)blockIdx.z * a.seg + cs) * a.H + h) * U::SIZE;
    const float d = DELTA ? 0.f : a.decay[h];

    // the tokens' vectors, activated; tokens past the end leave the state alone (w = 1, the others 0)
#pragma unroll
    for (int i = 0; i < C / 4; ++i) {
        const int tt = wave + 4 * i;
        const bool on = tt < nc;
        const size_t t = (size_t)(t0 + (on ? tt : 0));
        float r[EK], k[EK];
#pragma unroll
        for (int e = 0; e < EK; ++e) {
            const int idx = e * 64 + lane;
            const bool in = on && idx < DK;
            r[e] = in ? bf16_to_f32(a.r[t * a.r_stride + h * DK + idx]) : 0.f;
            k[e] = in ? bf16_to_f32(a.k[t * a.k_stride + h * DK + idx]) : 0.f;
        }
        if (DELTA) {
            float ssq = 0.f;
#pragma unroll
            for (int e = 0; e < EK; ++e) ssq = fmaf(k[e], k[e], ssq);
            const float inv = 1.f / sqrtf(wave_sum(ssq) + a.unit_eps);
#pragma unroll
            for (int e = 0; e < EK; ++e) {
                const int idx = e * 64 + lane;
                if (idx >= DK) continue;
                const int ch = h * DK + idx;
                const float u = on ? k[e] * inv : 0.f;       // (with a unit_eps of 0 a token past the end would make it 0 * inf)
                Um[tt * KP + idx] = u;
                Bm[tt * KP + idx] = on ? sigmoid_(bf16_to_f32(a.al[t * a.al_stride + ch]) + a.ab[ch]) * u : 0.f;
                Ws[tt * DK + idx] = on ? __expf(-a.decay_c * sigmoid_(bf16_to_f32(a.wl[t * a.wl_stride + ch]) + a.w0[ch])) : 1.f;
            }
        } else {
            if (a.silu_in) {
#pragma unroll
                for (int e = 0; e < EK; ++e) { r[e] = silu_(r[e]); k[e] = silu_(k[e]); }
            }
            if (a.rot_cos && on) {
                const int half = a.rot >> 1;
                const size_t pos = (size_t)(a.q_start[b] + c * C + tt);
#pragma unroll
                for (int e = 0; e < EK; ++e) {
                    const int idx = e * 64 + lane;
                    if (idx >= a.rot || idx >= DK) continue;
                    const bool low = idx < half;
                    const int j = low ? idx : idx - half, other = h * DK + (low ? idx + half : idx - half);
                    const float cs_ = a.rot_cos[pos * half + j], sn = low ? -a.rot_sin[pos * half + j] : a.rot_sin[pos * half + j];
                    r[e] = fmaf(bf16_to_f32(a.r[t * a.r_stride + other]), sn, r[e] * cs_);
                    k[e] = fmaf(bf16_to_f32(a.k[t * a.k_stride + other]), sn, k[e] * cs_);
                }
            }
#pragma unroll
            for (int e = 0; e < EK; ++e) k[e] *= a.k_scale;
        }
#pragma unroll
        for (int e = 0; e < EK; ++e) {
            const int idx = e * 64 + lane;
            if (idx < DK) { Rm[tt * KP + idx] = r[e]; Km[tt * KP + idx] = k[e]; }
        }
        for (int idx = lane; idx < DV; idx += 64) {
            float v = on ? bf16_to_f32(a.v[t * a.v_stride + h * DV + idx]) : 0.f;
            if (!DELTA && a.silu_in) v = silu_(v);
            Vm[tt * VP + idx] = v;
        }
    }
    if (!DELTA && tid <= C) Wc[tid] = power(d, tid);
    __syncthreads();
    if (DELTA) {
        // W up to each token: a wave has 8 tokens and multiplies those before them again
        constexpr int PER = C / 4;
#pragma unroll
        for (int e = 0; e < EK; ++e) {
            const int idx = e * 64 + lane;
            if (idx >= DK) continue;
            double p = 1.0;
            for (int tt = 0; tt < wave * PER; ++tt) p *= (double)Ws[tt * DK + idx];
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const int tt = wave * PER + i, at = tt * KP + idx;
                Um[at] = (float)((double)Um[at] * p);
                p *= (double)Ws[tt * DK + idx];
                const double inv = 1.0 / p;
                Rm[at] = (float)((double)Rm[at] * p);
                Km[at] = (float)((double)Km[at] * inv);
                Bm[at] = (float)((double)Bm[at] * inv);
            }
            if (wave == 3) Wc[idx] = p;
        }
        __syncthreads();
    }
    // the matrices of C x C, without the tile above the diagonal.  16 bytes of a row a lane make four steps of the
    // instruction.  Delta: a wave a matrix; else a wave a tile.
    {
        const float* X = !DELTA || (wave & 1) ? Rm : Um;
        const float* Y = !DELTA || wave < 2 ? Km : Bm;
        double* D = !DELTA || (wave & 1) ? A2 : T2;
        f64x4_t acc[3] = {};                                   // tiles (0, 0), (1, 0), (1, 1)
        const int p0 = !DELTA && wave > 0, q0 = !DELTA && wave > 1;    // the decay form's tile
        if (DELTA || wave < 3) {
#pragma unroll 2
            for (int j = 0; j < DK / 16; ++j) {
                float4 x[2], y[2];
#pragma unroll
                for (int q = 0; q < (DELTA ? 2 : 1); ++q) {
                    x[q] = *reinterpret_cast<const float4*>(X + (16 * (q + p0) + i16) * KP + 16 * j + 4 * g);
                    y[q] = *reinterpret_cast<const float4*>(Y + (16 * (q + q0) + i16) * KP + 16 * j + 4 * g);
                }
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const auto of = [&](const float4& v) { return (double)(s == 0 ? v.x : s == 1 ? v.y : s == 2 ? v.z : v.w); };
                    acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(of(x[0]), of(y[0]), acc[0], 0, 0, 0);
                    if (DELTA) {
                        acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(of(x[1]), of(y[0]), acc[1], 0, 0, 0);
                        acc[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(of(x[1]), of(y[1]), acc[2], 0, 0, 0);
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < (DELTA ? 3 : 1); ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int t = 16 * (DELTA ? i > 0 : p0) + 4 * e + g, s = 16 * (DELTA ? i > 1 : q0) + i16;
                    if (!DELTA) { if (s <= t) D[t * TP + s] = acc[i][e] * Wc[t - s]; }
                    else if (wave == 1) { if (s <= t) D[t * TP + s] = acc[i][e]; }               // A_k
                    else if (wave == 2) { if (s < t) D[t * TP + s] = acc[i][e]; }                // L
                    else if (s < t || (wave == 3 && s == t)) D[s * TP + t + 1] = acc[i][e];      // N, A_b
                }
        }
    }
    __syncthreads();
    if (DELTA) {
        // T = (I + L)^-1, a column a lane
        if (wave == 0) {
            const int j = lane & 31;
            double x[C], row[2][C];
#pragma unroll
            for (int t = 0; t < C; ++t) {
                if (t + 1 < C) {
#pragma unroll
                    for (int q = 0; q <= t; ++q) row[(t + 1) & 1][q] = T2[(t + 1) * TP + q];
                }
                double s[4] = {t == j ? 1.0 : 0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int q = 0; q < t; ++q) s[q & 3] = fma(-row[t & 1][q], x[q], s[q & 3]);
                x[t] = (s[0] + s[1]) + (s[2] + s[3]);
                asm volatile("" : "+v"(x[t]) :: "memory");       // one row of L ahead of its use, not all of them (registers)
            }
#pragma unroll
            for (int t = 0; t < C; ++t)
                if (t >= j) T2[t * TP + j] = x[t];
        }
        __syncthreads();
        // P = A_b T in the place of A_b: the first wave, which reads all of it before it writes.  The others G = T^T B~ ..
        constexpr int UNITS = 2 * (DK / 16), MINE = (UNITS + 2) / 3;       // tiles of [C][DK], of one of three waves
        if (wave == 0) {
            f64x4_t x[3] = {};
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const int t = 16 * (i > 0) + i16, col = 16 * (i > 1) + i16;
                const auto ab = [&](int s) { return second_of(A2, t, s); };
                const auto ts = [&](int s) { return first_of(T2, s, col); };
                x[i] = i == 0 ? product<0, 4>(x[i], g, ab, ts) : i == 1 ? product<0, 8>(x[i], g, ab, ts) : product<4, 8>(x[i], g, ab, ts);
            }
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int t = 16 * (i > 0) + 4 * e + g, s = 16 * (i > 1) + i16;
                    if (s <= t) A2[s * TP + t + 1] = x[i][e];
                }
        } else {
            for (int u = wave - 1; u < UNITS; u += 3) {
                const int half = u & 1, ch = (u >> 1) * 16 + i16;
                const double wc = Wc[ch];
                const auto ts = [&](int s) { return first_of(T2, s, 16 * half + i16); };
                const auto bs = [&](int s) { return (double)Bm[s * KP + ch] * wc; };
                f64x4_t x = {};
                x = half ? product<4, 8>(x, g, ts, bs) : product<0, 8>(x, g, ts, bs);
#pragma unroll
                for (int e = 0; e < 4; ++e) Gs[(16 * half + 4 * e + g) * HP + ch] = x[e];
            }
        }
        __syncthreads();
        // .. then E = A_k - P N in the place of A_k, and H = K~ - N^T G
        f64x4_t hs[MINE];
        if (wave == 0) {
            f64x4_t x[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const int t = 16 * (i > 0) + i16, col = 16 * (i > 1) + i16;
#pragma unroll
                for (int e = 0; e < 4; ++e) x[i][e] = first_of(A2, 16 * (i > 0) + 4 * e + g, col);
                const auto ps = [&](int s) { return -second_of(A2, t, s); };
                const auto ns = [&](int s) { return second_strictly(T2, s, col); };
                x[i] = i == 0 ? product<0, 4>(x[i], g, ps, ns) : i == 1 ? product<0, 8>(x[i], g, ps, ns) : product<4, 8>(x[i], g, ps, ns);
            }
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int t = 16 * (i > 0) + 4 * e + g, s = 16 * (i > 1) + i16;
                    if (s <= t) A2[t * TP + s] = x[i][e];
                }
        } else {
#pragma unroll
            for (int m = 0; m < MINE; ++m) {
                const int u = min(wave - 1 + 3 * m, UNITS - 1), half = u & 1, ch = (u >> 1) * 16 + i16;
                const double wc = Wc[ch];
#pragma unroll
                for (int e = 0; e < 4; ++e) hs[m][e] = (double)Km[(16 * half + 4 * e + g) * KP + ch] * wc;
                const auto ns = [&](int s) { return -second_strictly(T2, s, 16 * half + i16); };
                const auto gs = [&](int s) { return Gs[s * HP + ch]; };
                hs[m] = half ? product<4, 8>(hs[m], g, ns, gs) : product<0, 8>(hs[m], g, ns, gs);
            }
        }
        __syncthreads();
        if (wave > 0) {
#pragma unroll
            for (int m = 0; m < MINE; ++m) {
                const int u = wave - 1 + 3 * m, half = u & 1, ch = (u >> 1) * 16 + i16;
                if (u >= UNITS) continue;
#pragma unroll
                for (int e = 0; e < 4; ++e) Hs[(16 * half + 4 * e + g) * HP + ch] = hs[m][e];
            }
        }
        __syncthreads();
    }
    bool bad = false;
    const auto rounded = [&](const f64x4_t& x) {
        const float4 y = make_float4((float)x[0], (float)x[1], (float)x[2], (float)x[3]);
        bad |= endless(y.x) || endless(y.y) || endless(y.z) || endless(y.w);
        return y;
    };
    const auto place = [&](int from, int tile) { return reinterpret_cast<float4*>(unit + from) + tile * 64 + lane; };
    // R' transposed (rows: channels, columns: tokens)
    for (int kt = wave; kt < DK / 16; kt += 4) {
        const auto us = [&](int s) { return -(double)Um[s * KP + kt * 16 + turned(i16)]; };
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int t = 16 * half + i16;
            const float4 r4 = *reinterpret_cast<const float4*>(Rm + t * KP + kt * 16 + 4 * g);
            f64x4_t x = {(double)r4.x, (double)r4.y, (double)r4.z, (double)r4.w};
            if (DELTA) {
                const auto ps = [&](int s) { return second_of(A2, t, s); };
                x = half ? product<0, 8>(x, g, us, ps) : product<0, 4>(x, g, us, ps);
            } else {
                const double w = Wc[t + 1];
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] *= w;
            }
            *place(U::R, half * (DK / 16) + kt) = rounded(x);
        }
    }
    // the chunk's own part of the outputs
    for (int ct = (wave + 2) & 3; ct < DV / 16; ct += 4) {
        const auto vs = [&](int s) { return (double)Vm[s * VP + ct * 16 + i16]; };
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const auto es = [&](int s) { return first_of(A2, 16 * half + i16, s); };
            f64x4_t x = {};
            x = half ? product<0, 8>(x, g, es, vs) : product<0, 4>(x, g, es, vs);
            const float4 y = rounded(x);
            const float ye[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = 16 * half + 4 * e + g;
                if (t < nc) a.out[(size_t)(t0 + t) * a.out_stride + h * DV + ct * 16 + i16] = ye[e];
            }
        }
    }
    // 32 x 32 results: rows of A's channels, columns of B's
    const auto square = [&](int from, int rows, int cols, int rt, int ct, auto fa, auto fb) {
        f64x4_t x[2][2] = {};
#pragma unroll
        for (int s = 0; s < C / 4; ++s) {
            double p[2], q[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) { p[i] = fa(4 * s + g, (2 * rt + i) * 16 + turned(i16)); q[i] = fb(4 * s + g, (2 * ct + i) * 16 + i16); }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) x[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(p[i], q[j], x[i][j], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) *place(from, (2 * ct + j) * (rows / 16) + 2 * rt + i) = rounded(x[i][j]);
    };
    // what the chunk adds to the state
    for (int m = wave; m < TK * TV; m += 4) {
        const auto vs = [&](int t, int col) { return (double)Vm[t * VP + col]; };
        if (DELTA) square(U::S, DK, DV, m / TV, m % TV, [&](int t, int ch) { return Hs[t * HP + ch]; }, vs);
        else square(U::S, DK, DV, m / TV, m % TV, [&](int t, int ch) { return (double)Km[t * KP + ch] * Wc[max(nc - 1 - t, 0)]; }, vs);   // (k is zero past the end)
    }
    if (DELTA) {
        // M transposed (rows: the channel it is summed over, columns: the channel it goes to), without W_C on its diagonal
        for (int m = wave; m < TK * TK; m += 4)
            square(U::M, DK, DK, m / TK, m % TK, [&](int t, int ch) { return -(double)Um[t * KP + ch]; }, [&](int t, int ch) { return Gs[t * HP + ch]; });
        if (tid < DK) {
            const float w = (float)Wc[tid];
            unit[U::W + tid] = w;
            bad |= endless(w);
        }
    }
    const int any = __syncthreads_or(bad);
    if (tid == 0) reinterpret_cast<int*>(unit)[U::BAD] = any;
}

// The state through the segment's chunks, 16 of its columns a block.  A wave owns 32 rows (two tiles of 16); with
// v_mfma_f32_16x16x4_f32 a result (row 4 g + i, column l % 16 in element i of lane 16 g + l % 16) is the operand of
// the next product as it lies, for the four k values {16 a + 4 g + i}: the operators are stored for that order.  The
// waves hand their rows to each other through LDS.
// Tiles of 16 key rows of the state a wave: one where a chunk's operators fit two waves more beside each other, us a layer of 2,048
// tokens, 32 heads of 64, two tiles / one: delta form 101 / 86; the decay form, whose waves then no longer all have outputs, 55 / 69.
constexpr int state_tiles(int dk, bool delta) { return delta && dk <= 64 ? 1 : 2; }

// D: chunks whose operands are under way.
template <int DK, int DV, bool DELTA, int D>
__global__ __launch_bounds__(DK * 4 / state_tiles(DK, DELTA)) void chunk_states_kernel(const ChunkArgs a) {
    constexpr int Q = state_tiles(DK, DELTA), NA = DK / 16, NW = NA / Q;
    using U = Unit<DK, DV, DELTA>;
    const int b = a.rows ? a.rows[blockIdx.z] : (int)blockIdx.z, h = blockIdx.x, cb = blockIdx.y;
    if (b < 0) return;
    const int t_lo = a.cu_q[b], n = a.cu_q[b + 1] - t_lo;
    if (n < a.min_tokens || a.c0 * C >= n) return;
    int* const from = a.from + ((size_t)b * a.H + h) * (DV / 16) + cb;       // (this block's own, the same in all of a head's)
    if (a.c0 > 0 && *from < a.c0 * C) return;          // the walk takes the row over before this segment
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), col = lane & 15, g = lane >> 4;
    const int all = min(a.seg, (n + C - 1) / C - a.c0);          // at most 64
    const float* units = a.ws + ((size_t)blockIdx.z * a.seg * a.H + h) * U::SIZE;
    const unsigned long long bads = __ballot(lane < all && reinterpret_cast<const int*>(units + (size_t)lane * a.H * U::SIZE)[U::BAD] != 0);
    const int chunks = bads ? __ffsll(bads) - 1 : all;
    if (threadIdx.x == 0) *from = (a.c0 + chunks) * C;
    __shared__ __align__(16) f32x4_t St[2][NA][64];
    float* Sg = a.state + ((size_t)a.slots[b] * a.H + h) * (size_t)DK * DV + cb * 16 + col;
    const bool fresh = a.c0 == 0 && a.q_start[b] == 0;
    f32x4_t S[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) S[q][i] = fresh ? 0.f : Sg[(size_t)((wave * Q + q) * 16 + 4 * g + i) * DV];
    struct Ops { f32x4_t m[DELTA ? Q : 1][DELTA ? NA : 1], w[DELTA ? Q : 1], r[NA], add[Q], o; };
    const bool outputs = NW == 2 || wave < 2;    // two tiles of 16 tokens
    const float d = DELTA ? 0.f : a.decay[h];
    const double d_chunk = DELTA ? 0.0 : power(d, C);
    auto ask = [&](int c, Ops& x) {
        const f32x4_t* unit = reinterpret_cast<const f32x4_t*>(units + (size_t)c * a.H * U::SIZE);
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            x.add[q] = unit[U::S / 4 + (cb * NA + wave * Q + q) * 64 + lane];
            if (DELTA) {
#pragma unroll
                for (int k = 0; k < NA; ++k) x.m[q][k] = unit[U::M / 4 + ((wave * Q + q) * NA + k) * 64 + lane];
                x.w[q] = unit[U::W / 4 + (wave * Q + q) * 4 + g];
            }
        }
        if (outputs) {
#pragma unroll
            for (int k = 0; k < NA; ++k) x.r[k] = unit[U::R / 4 + (wave * NA + k) * 64 + lane];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = min((a.c0 + c) * C + wave * 16 + 4 * g + i, n - 1);          // what lies behind the last token is not stored
                x.o[i] = a.out[(size_t)(t_lo + t) * a.out_stride + h * DV + cb * 16 + col];
            }
        }
    };
    auto step = [&](int c, Ops& x) {
#pragma unroll
        for (int q = 0; q < Q; ++q) St[c & 1][wave * Q + q][lane] = S[q];
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // LDS only: the next chunk's loads stay under way
        const double dc = DELTA ? 0.0 : ((a.c0 + c + 1) * C <= n ? d_chunk : power(d, n - (a.c0 + c) * C));
        // the instruction adds in order: short chains, for the outputs of 8 or 16 products
        constexpr int CH = 4, CO = 8;
        f32x4_t next[Q][CH] = {}, o[CO] = {};
#pragma unroll
        for (int k = 0; k < NA; ++k) {
            const f32x4_t s = St[c & 1][k][lane];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (DELTA) {
#pragma unroll
                    for (int q = 0; q < Q; ++q)
                        next[q][(4 * k + i) % CH] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.m[q][k][i], s[i], next[q][(4 * k + i) % CH], 0, 0, 0);
                }
                if (outputs) o[(4 * k + i) % CO] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.r[k][i], s[i], o[(4 * k + i) % CO], 0, 0, 0);
            }
        }
        if (outputs) {
            const f32x4_t whole = ((o[0] + o[1]) + (o[2] + o[3])) + ((o[4] + o[5]) + (o[6] + o[7]));
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = (a.c0 + c) * C + wave * 16 + 4 * g + i;
                if (t < n) a.out[(size_t)(t_lo + t) * a.out_stride + h * DV + cb * 16 + col] = x.o[i] + whole[i];
            }
        }
        // the new state, rounded once
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const f32x4_t whole = (next[q][0] + next[q][1]) + (next[q][2] + next[q][3]);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                S[q][i] = DELTA ? (float)(fma((double)x.w[q][i], (double)S[q][i], (double)x.add[q][i]) + (double)whole[i])
                                : (float)fma(dc, (double)S[q][i], (double)x.add[q][i]);
        }
    };
    static_assert(NW >= 2, "two waves make the outputs");
    // D chunks' operands under way, asked for under no condition (the last one's again behind the end): at a place that can be
    // reached with fewer loads under way the compiled code would wait for more of them.
    Ops x[D];
    if (chunks > 0) {
#pragma unroll
        for (int d = 0; d < D; ++d) ask(min(d, chunks - 1), x[d]);
        int c = 0;
        for (; c + D <= chunks; c += D)
#pragma unroll
            for (int d = 0; d < D; ++d) {
                step(c + d, x[d]);
                ask(min(c + d + D, chunks - 1), x[d]);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
        for (int d = 0; d < D - 1; ++d)
            if (c + d < chunks) step(c + d, x[d]);
    }
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) Sg[(size_t)((wave * Q + q) * 16 + 4 * g + i) * DV] = S[q][i];
}

template <int DK, int DV, bool DELTA>
int launch_chunks(ChunkArgs a, int rows, int max_tokens, hipStream_t stream) {
    constexpr size_t lds = sizeof(float) * Lds<DK, DV, DELTA>::SIZE;
    static_assert(lds <= 160 * 1024 && (DK > 64 || lds <= 80 * 1024), "more LDS than a compute unit has, or than half of it");
    auto operators = chunk_operators_kernel<DK, DV, DELTA>;
    if (lds > 64 * 1024) {          // beyond what a kernel may take unasked: ask once a device
        static std::mutex mu;
        static bool asked[64] = {};
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        RI_REQUIRE(e == hipSuccess && dev >= 0 && dev < 64, "ri_linear_scan_chunks: no current device: %s", hipGetErrorString(e));
        std::lock_guard<std::mutex> lock(mu);
        if (!asked[dev]) {
            e = hipFuncSetAttribute(reinterpret_cast<const void*>(operators), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            RI_REQUIRE(e == hipSuccess, "ri_linear_scan_chunks: %zu bytes of LDS refused: %s", lds, hipGetErrorString(e));
            asked[dev] = true;
        }
    }
    const int chunks = (max_tokens + C - 1) / C;
    for (a.c0 = 0; a.c0 < chunks; a.c0 += a.seg) {
        operators<<<dim3(min(a.seg, chunks - a.c0), a.H, rows), 256, lds, stream>>>(a);
        // a head on one XCD: its blocks read the same operators.  Four chunks under way, of heads of 128 two, and three of a single row in the decay form,
        // us, two / three: 24 heads, 2,048 tokens 195 / 182 (190 with loads that the compiled loop waited for), 300 51.6 / 50.2; rows of 200, two 59.7 / 65.2, three 70 / 77
        auto states = chunk_states_kernel<DK, DV, DELTA, DK <= 64 ? 4 : 2>;
        if constexpr (DK > 64 && !DELTA) if (rows == 1) states = chunk_states_kernel<DK, DV, DELTA, 3>;
        states<<<dim3(a.H, DV / 16, rows), DK * 4 / state_tiles(DK, DELTA), 0, stream>>>(a);
    }
    return 0;
}

// chunks of each of so many rows that one pass takes: the workspace holds some 64 chunks of all heads
int segment(int rows, int max_tokens) {
    const int chunks = (max_tokens + C - 1) / C, most = rows < 64 ? 64 / rows : 1;
    return chunks < most ? chunks : most;
}

}  // namespace

// Whether ri_linear_scan_chunks takes heads of this size (delta: with decays of at least exp(-decay_c)).
extern "C" int ri_linear_scan_chunks_supported(int delta, int dk, int dv, float decay_c) {
    if (delta && !(decay_c >= 0.f && decay_c * C <= 60.f)) return 0;      // W_C >= 1e-26
    return (dk == 64 || dk == 128) && dv == dk;
}

static size_t unit_floats(int delta, int rows, int max_tokens, int H, int dk, int dv) {
    return (size_t)rows * segment(rows, max_tokens) * H * ((size_t)C * dk + (size_t)dk * dv + (delta ? (size_t)dk * dk + dk : 0) + 4);
}

// Floats of workspace that are enough for any step of at most num_rows rows: 64 chunks of all heads, whatever the number
// and length of its portions up to 64 of them.
extern "C" size_t ri_linear_scan_chunks_workspace(int delta, int num_rows, int H, int dk, int dv) {
    return unit_floats(delta, 1, 64 * C, H, dk, dv) + (size_t)num_rows * H * (dv / 16);
}

extern "C" int ri_linear_scan(
        const void* r, int r_stride, const void* k, int k_stride, const void* v, int v_stride,
        const void* wl, int wl_stride, const void* al, int al_stride, int dtype,
        const float* w0, const float* ab, const float* decay, int delta, int silu_in,
        float unit_eps, float decay_c, float* state, int num_slots, float* out, int out_stride,
        const int* cu_q, const int* q_start, const int* slots, int num_rows, int T,
        int H, int dk, int dv, const float* rot_cos, const float* rot_sin, int rot, int rot_rows, int max_position,
        float k_scale, int most, const int* from, int from_cols, hipStream_t stream);

// ri_linear_scan with the rows of at least min_tokens tokens (max_tokens at most, or an upper bound) in chunks; the walk
// does the others, and what the chunks leave to it.  row_list [listed]: the rows of several tokens, then -1, which must
// hold all rows of min_tokens and more; a pass, its grid and the workspace are theirs, however many rows of
// single tokens the step has (null: all rows, listed = num_rows).  bfloat16 projections.
extern "C" int ri_linear_scan_chunks(
        const void* r, int r_stride, const void* k, int k_stride, const void* v, int v_stride,
        const void* wl, int wl_stride, const void* al, int al_stride,
        const float* w0, const float* ab, const float* decay, int delta, int silu_in,
        float unit_eps, float decay_c, float* state, int num_slots, float* out, int out_stride,
        const int* cu_q, const int* q_start, const int* slots, int num_rows, int T,
        int H, int dk, int dv, const float* rot_cos, const float* rot_sin, int rot, int rot_rows, int max_position,
        float k_scale, int min_tokens, int max_tokens, const int* row_list, int listed, float* ws, size_t ws_floats, hipStream_t stream) {
    RI_REQUIRE(H > 0 && ri_linear_scan_chunks_supported(delta, dk, dv, decay_c), "ri_linear_scan_chunks: does not take H=%d dk=%d dv=%d decay_c=%g", H, dk, dv, (double)decay_c);
    RI_REQUIRE(num_rows >= 0 && T >= 0 && num_slots > 0 && min_tokens > 1 && (row_list ? listed >= 0 && listed <= num_rows : listed == num_rows), "ri_linear_scan_chunks: bad counts");
    RI_REQUIRE(r_stride >= H * dk && k_stride >= H * dk && v_stride >= H * dv && out_stride >= H * dv, "ri_linear_scan_chunks: row strides too small");
    if (num_rows == 0 || T == 0) return 0;
    RI_REQUIRE(listed > 0 && max_tokens > 0, "ri_linear_scan_chunks: no row of several tokens");
    RI_REQUIRE(r && k && v && state && out && cu_q && q_start && slots && ws, "ri_linear_scan_chunks: null pointer");
    RI_REQUIRE(H <= 65535 && num_rows <= 65535, "ri_linear_scan_chunks: too many heads or rows for the grid");
    RI_REQUIRE((uintptr_t)ws % 16 == 0 && ws_floats >= unit_floats(delta, listed, max_tokens, H, dk, dv) + (size_t)num_rows * H * (dv / 16), "ri_linear_scan_chunks: the workspace is too small");
    if (delta) RI_REQUIRE(wl && al && w0 && ab && wl_stride >= H * dk && al_stride >= H * dk && !rot_cos && k_scale == 1.f, "ri_linear_scan_chunks: the delta form needs wl, al, w0, ab and no rotation or key factor");
    else RI_REQUIRE(decay, "ri_linear_scan_chunks: the decay form needs a decay for each head");
    if (rot_cos) RI_REQUIRE(!silu_in && rot_sin && rot > 0 && rot % 2 == 0 && rot <= dk && rot_rows > 0 && max_position < rot_rows,
                            "ri_linear_scan_chunks: a rotation goes without silu, an even rot <= dk and tables of %d positions (got %d rows)", max_position + 1, rot_rows);
    ChunkArgs a;
    a.r = (const bf16_t*)r; a.k = (const bf16_t*)k; a.v = (const bf16_t*)v; a.wl = (const bf16_t*)wl; a.al = (const bf16_t*)al;
    a.r_stride = r_stride; a.k_stride = k_stride; a.v_stride = v_stride; a.wl_stride = wl_stride; a.al_stride = al_stride;
    a.w0 = w0; a.ab = ab; a.decay = decay; a.state = state; a.out = out; a.out_stride = out_stride;
    a.cu_q = cu_q; a.q_start = q_start; a.slots = slots; a.H = H; a.silu_in = silu_in; a.min_tokens = min_tokens;
    a.unit_eps = unit_eps; a.decay_c = decay_c; a.rot_cos = rot_cos; a.rot_sin = rot_sin; a.rot = rot_cos ? rot : 0; a.k_scale = k_scale;
    a.rows = row_list; a.ws = ws; a.c0 = 0; a.seg = segment(listed, max_tokens);
    a.from = reinterpret_cast<int*>(ws + unit_floats(delta, listed, max_tokens, H, dk, dv));
    int rc;
    if (dk == 64) rc = delta ? launch_chunks<64, 64, true>(a, listed, max_tokens, stream) : launch_chunks<64, 64, false>(a, listed, max_tokens, stream);
    else rc = delta ? launch_chunks<128, 128, true>(a, listed, max_tokens, stream) : launch_chunks<128, 128, false>(a, listed, max_tokens, stream);
    if (rc) return rc;
    RI_LAUNCHED("ri_linear_scan_chunks");
    return ri_linear_scan(r, r_stride, k, k_stride, v, v_stride, wl, wl_stride, al, al_stride, RI_BF16, w0, ab, decay, delta, silu_in,
                          unit_eps, decay_c, state, num_slots, out, out_stride, cu_q, q_start, slots, num_rows, T, H, dk, dv,
                          rot_cos, rot_sin, rot, rot_rows, max_position, k_scale, min_tokens - 1, a.from, dv / 16, stream);
}
