// The state walk of recurrent.hip for prompts, 32 tokens at a time on the 32-bit matrix instructions:
//
//   delta form:  S_t = diag(w_t) S_(t-1) - b_t (u_t^T S_(t-1)) + k_t v_t^T,   o_t = S_t^T r_t
//   decay form:  S_t = d S_(t-1) + k_t v_t^T,                                 o_t = S_t^T r_t
//
// per head, S of [dk][dv], b = a * u.  Token by token that is a chain of thousands of short steps on a quarter of
// the chip's SIMDs.  Within a chunk of C tokens, with W_t = w_1 * .. * w_t (per key channel) and
//   U_t = u_t W_(t-1),   R_t = r_t W_t,   K_t = k_t / W_t,   B_t = b_t / W_t,
// the tokens' d_t = u_t^T S_(t-1) solve (I + L) D = U S_0 + N V with L, N the strictly lower parts of U B^T and U K^T,
// so D = X S_0 + Y V' with X, Y from one substitution on [U | N V], and
//   o   = (R - A_b X) S_0 + (A_k V - A_b Y),      A_k, A_b the lower parts of R K^T, R B^T
//   S_C = (diag(W_C) - B~^T X) S_0 + (K~^T V - B~^T Y),      K~ = K W_C, B~ = B W_C.
// Everything but S_0 is the chunk's own: `chunk_operators_kernel` makes it for all chunks at once (a block a
// chunk and head), and `chunk_states_kernel` passes the state through the chunks: one product of dk x dk and one of
// C x dk against 16 of its columns a block.  The decay form has powers of d in place of the operators.
//
// W only ever divides what is multiplied by a later W: a ratio W_t / W_s is as exact as the product of the decays
// between, however small both are.  That needs W_C > 0: the caller takes this form where the design bounds the
// decays (w >= exp(-decay_c)).  A substitution and not a product of powers of L: where keys repeat, those grow
// beyond what cancels.  Sums are in chains of 8 or 16 products, and the
// delta form's W and its four C x C matrices in 64 bits: with single chains the outputs are two to three times
// further from 64-bit arithmetic than the walk's, so they are as close (1.0e-7; the decay form 1.2e-7 against 2.6e-7).
//
// What holds the tokens of a chunk apart is zeros, which a value that is not finite passes.  A chunk and head whose operators
// are not finite (a token's vectors were not, or k / W_t left the range of 32 bits) is therefore only marked; the states
// stop in front of it, and the walk does that head of that row from there on, so that every token gets what the walk gives.
//
// 2,048 tokens of 32 heads of 64, us a layer: delta form 1205 -> 232 (137 the operators, 95 the states), decay form
// 768 -> 100; 24 heads of 128: 1741 -> 559, 1011 -> 174.  The operators are bound by the steps of a block following
// each other (matrix instructions a quarter of the time, two blocks a compute unit), the states by the chain of chunks.
#include "common.h"
#include <mutex>

namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef double f64x4_t __attribute__((ext_vector_type(4)));

constexpr int C = 32;                   // tokens a chunk
constexpr int CP = C + 4;               // floats a row of a C x C matrix takes in LDS

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
    float* ws;                          // [row][chunk of the segment][head][Unit::SIZE]
    int* from;                          // [row][head][dv / 16]: the token that the walk goes on from
    int c0, seg;                        // the segment's first chunk of every row, its chunks
};

__device__ __forceinline__ float sigmoid_(float z) { return __fdividef(1.f, 1.f + __expf(-z)); }
__device__ __forceinline__ float silu_(float z) { return __fdividef(z, 1.f + __expf(-z)); }

// Floats of a chunk and head in the workspace: R' [2 tiles of 16 tokens][dk / 16][64][4], S_add [dv / 16][dk / 16][64][4]
// and, in the delta form, M [dk / 16][dk / 16][64][4]: each in the order the lanes of chunk_states_kernel read it; BAD: not
// zero where something in it is not finite.
template <int DK, int DV, bool DELTA>
struct Unit {
    static constexpr int R = 0, S = C * DK, M = S + DK * DV, BAD = M + (DELTA ? DK * DK : 0), SIZE = BAD + 4;
};
__device__ __forceinline__ bool endless(float x) { return !(fabsf(x) < __builtin_inff()); }

// d to the power n (0 <= n <= C), rounded once
__device__ __forceinline__ float power(float d, int n) {
    double p = 1.0, q = (double)d;
    for (int m = n; m > 0; m >>= 1) {
        if (m & 1) p *= q;
        q *= q;
    }
    return (float)p;
}

// acc += A B over the C tokens of a chunk, two a matrix instruction: a lane's operands are rows / columns l % 32,
// token 2 s + l / 32.  Four chains of sums: the instruction adds in order, and one chain of 32 or 64 products is
// two to three times further from the exact sum than the walk's eight-row sums are.
template <typename FA, typename FB>
__device__ __forceinline__ f32x16_t product(f32x16_t acc, FA a, FB b) {
    f32x16_t p[4] = {};
#pragma unroll
    for (int s = 0; s < C / 2; ++s) p[s & 3] = __builtin_amdgcn_mfma_f32_32x32x2f32(a(s), b(s), p[s & 3], 0, 0, 0);
    return acc + ((p[0] + p[1]) + (p[2] + p[3]));
}
// rows of a 32 x 32 result in element e of a lane: 8 (e / 4) + 4 (l / 32) + e % 4; column l % 32

template <int DK, int DV, bool DELTA>
__global__ __launch_bounds__(256) void chunk_operators_kernel(const ChunkArgs a) {
    constexpr int KP = DK + 4, VP = DV + 4, NX = DELTA ? DK + DV : 0, XP = NX + 4;
    constexpr int EK = DK / 64 > 0 ? DK / 64 : 1, TK = DK / 32, TV = DV / 32;
    using U = Unit<DK, DV, DELTA>;
    const int b = blockIdx.z, h = blockIdx.y, cs = blockIdx.x, c = a.c0 + cs;
    const int t_lo = a.cu_q[b], n = a.cu_q[b + 1] - t_lo;
    if (n < a.min_tokens || c * C >= n) return;
    const int nc = min(C, n - c * C), t0 = t_lo + c * C;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, hi = lane >> 5;
    extern __shared__ __align__(16) float lds[];
    float* Rm = lds;                          // [C][KP]: r, then R
    float* Km = Rm + C * KP;                  // k, then K
    float* Vm = Km + C * KP;                  // [C][VP]
    float* Ak = Vm + C * VP;                  // [C][CP]
    float* Wc = Ak + C * CP;                  // [DK]: W_C; the decay form: powers of d, 0 .. C
    float* Um = Wc + (DK > C + 4 ? DK : C + 4);       // delta: u, then U
    float* Bm = Um + C * KP;                  // b, then B
    float* Lm = Bm + C * KP;                  // [C][CP]
    float* Nm = Lm + C * CP;
    float* Ab = Nm + C * CP;
    float* Xm = Ab + C * CP;                  // [C][XP]: w first, then [U | N V], then [X | Y]
    float* unit = a.ws + (((size_t)b * a.seg + cs) * a.H + h) * U::SIZE;
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
                Xm[tt * XP + idx] = on ? __expf(-a.decay_c * sigmoid_(bf16_to_f32(a.wl[t * a.wl_stride + ch]) + a.w0[ch])) : 1.f;
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
        // W up to each token: a wave has 8 tokens and multiplies those before them again; the products first, in
        // registers, because the rows of w are where [U | N V] goes
        constexpr int PER = C / 4;
        double wt[EK][PER + 1];                // W before the wave's first token, then after each (64-bit: each factor is rounded once)
#pragma unroll
        for (int e = 0; e < EK; ++e) {
            const int idx = min(e * 64 + lane, DK - 1);
            double p = 1.0;
            for (int tt = 0; tt < wave * PER; ++tt) p *= (double)Xm[tt * XP + idx];
            wt[e][0] = p;
#pragma unroll
            for (int i = 0; i < PER; ++i) { p *= (double)Xm[(wave * PER + i) * XP + idx]; wt[e][i + 1] = p; }
            if (wave == 3 && e * 64 + lane < DK) Wc[idx] = (float)p;
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < EK; ++e) {
            const int idx = e * 64 + lane;
            if (idx >= DK) continue;
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const int at = (wave * PER + i) * KP + idx;
                const double inv = 1.0 / wt[e][i + 1];
                const float U_ = (float)((double)Um[at] * wt[e][i]);
                Um[at] = U_;
                Xm[(wave * PER + i) * XP + idx] = U_;
                Rm[at] = (float)((double)Rm[at] * wt[e][i + 1]);
                Km[at] = (float)((double)Km[at] * inv);
                Bm[at] = (float)((double)Bm[at] * inv);
            }
        }
        __syncthreads();
    }
    // the four matrices of C x C: a wave each (the decay form: the first wave)
    if (DELTA || wave == 0) {
        const float* X = !DELTA || (wave & 1) ? Rm : Um;
        const float* Y = !DELTA || wave < 2 ? Km : Bm;
        float* D = !DELTA ? Ak : (wave == 0 ? Nm : wave == 1 ? Ak : wave == 2 ? Lm : Ab);
        const bool strict = DELTA && !(wave & 1);
        if (DELTA) {
            // in 64 bits (v_mfma_f64_16x16x4_f64: lane 16 g + i has row or column i and one of four k; 16 bytes of K a lane
            // make four steps): what the substitution starts from decides how exact the chunk is
            const int i16 = lane & 15, g = lane >> 4;
            f64x4_t acc[2][2] = {};
#pragma unroll 2
            for (int j = 0; j < DK / 16; ++j) {
                float4 x[2], y[2];
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    x[q] = *reinterpret_cast<const float4*>(X + (16 * q + i16) * KP + 16 * j + 4 * g);
                    y[q] = *reinterpret_cast<const float4*>(Y + (16 * q + i16) * KP + 16 * j + 4 * g);
                }
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int p = 0; p < 2; ++p)
#pragma unroll
                        for (int q = 0; q < 2; ++q)
                            acc[p][q] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)(s == 0 ? x[p].x : s == 1 ? x[p].y : s == 2 ? x[p].z : x[p].w),
                                                                             (double)(s == 0 ? y[q].x : s == 1 ? y[q].y : s == 2 ? y[q].z : y[q].w), acc[p][q], 0, 0, 0);
            }
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int t = 16 * p + 4 * e + g, s = 16 * q + i16;
                        D[t * CP + s] = (strict ? s < t : s <= t) ? (float)acc[p][q][e] : 0.f;
                    }
        } else {
            f32x16_t p[4] = {};
#pragma unroll
            for (int j = 0; j < DK / 8; ++j) {
                const float4 x = *reinterpret_cast<const float4*>(X + l32 * KP + 8 * j + 4 * hi);
                const float4 y = *reinterpret_cast<const float4*>(Y + l32 * KP + 8 * j + 4 * hi);
                p[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(x.x, y.x, p[0], 0, 0, 0);
                p[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(x.y, y.y, p[1], 0, 0, 0);
                p[2] = __builtin_amdgcn_mfma_f32_32x32x2f32(x.z, y.z, p[2], 0, 0, 0);
                p[3] = __builtin_amdgcn_mfma_f32_32x32x2f32(x.w, y.w, p[3], 0, 0, 0);
            }
            const f32x16_t acc = (p[0] + p[1]) + (p[2] + p[3]);
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int t = 8 * (e >> 2) + 4 * hi + (e & 3);
                D[t * CP + l32] = l32 <= t ? acc[e] * Wc[t - l32] : 0.f;
            }
        }
    }
    __syncthreads();
    const auto lower = [&](const float* D) { return [=](int s) { return D[l32 * CP + 2 * s + hi]; }; };          // row l32
    const auto across = [&](const float* D, int stride, int at) { return [=](int s) { return D[(2 * s + hi) * stride + at + l32]; }; };
    if (DELTA) {
        // N V, where the substitution expects it
        for (int ct = wave; ct < TV; ct += 4) {
            const f32x16_t acc = product(f32x16_t{}, lower(Nm), across(Vm, VP, ct * 32));
#pragma unroll
            for (int e = 0; e < 16; ++e) Xm[(8 * (e >> 2) + 4 * hi + (e & 3)) * XP + DK + ct * 32 + l32] = acc[e];
        }
        __syncthreads();
        // (I + L) [X | Y] = [U | N V], a column a thread
        if (tid < NX) {
            float x[C];
#pragma unroll
            for (int t = 0; t < C; ++t) {
                float s = Xm[t * XP + tid];
#pragma unroll
                for (int q = 0; q < t; q += 4) {
                    const float4 l4 = *reinterpret_cast<const float4*>(Lm + t * CP + q);      // zeros from the diagonal on
                    s = fmaf(-l4.x, x[q], s);
                    if (q + 1 < t) s = fmaf(-l4.y, x[q + 1], s);
                    if (q + 2 < t) s = fmaf(-l4.z, x[q + 2], s);
                    if (q + 3 < t) s = fmaf(-l4.w, x[q + 3], s);
                }
                x[t] = s;
            }
#pragma unroll
            for (int t = 0; t < C; ++t) Xm[t * XP + tid] = x[t];
        }
        __syncthreads();
    }
    const auto minus = [](f32x16_t x) {
#pragma unroll
        for (int e = 0; e < 16; ++e) x[e] = -x[e];
        return x;
    };
    bool bad = false;
    const auto check = [&](const f32x16_t& x) {
#pragma unroll
        for (int e = 0; e < 16; ++e) bad |= endless(x[e]);
    };
    // R' transposed (rows: channels, columns: tokens), so that a lane's four consecutive rows are one store
    for (int it = wave; it < TK; it += 4) {
        f32x16_t acc;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int ch = it * 32 + 8 * (e >> 2) + 4 * hi + (e & 3);
            acc[e] = Rm[l32 * KP + ch] * (DELTA ? 1.f : Wc[l32 + 1]);
        }
        if (DELTA) acc = minus(product(minus(acc), across(Xm, XP, it * 32), lower(Ab)));
        check(acc);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int kt = it * 2 + (q >> 1), g = (q & 1) * 2 + hi;
            *reinterpret_cast<float4*>(unit + U::R + ((((l32 >> 4) * (DK / 16) + kt) * 64 + g * 16 + (l32 & 15)) * 4)) =
                make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
        }
    }
    // the chunk's own part of the outputs
    for (int ct = (wave + 2) & 3; ct < TV; ct += 4) {
        f32x16_t acc = {};
        if (DELTA) acc = minus(product(acc, lower(Ab), across(Xm, XP, DK + ct * 32)));
        acc = product(acc, lower(Ak), across(Vm, VP, ct * 32));
        check(acc);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int t = 8 * (e >> 2) + 4 * hi + (e & 3);
            if (t < nc) a.out[(size_t)(t0 + t) * a.out_stride + h * DV + ct * 32 + l32] = acc[e];
        }
    }
    // what the chunk adds to the state
    for (int m = wave; m < TK * TV; m += 4) {
        const int it = m / TV, ct = m % TV;
        const float wc = DELTA ? Wc[it * 32 + l32] : 0.f;
        f32x16_t acc = {};
        if (DELTA) {
            acc = minus(product(acc, [&](int s) { return Bm[(2 * s + hi) * KP + it * 32 + l32] * wc; }, across(Xm, XP, DK + ct * 32)));
            acc = product(acc, [&](int s) { return Km[(2 * s + hi) * KP + it * 32 + l32] * wc; }, across(Vm, VP, ct * 32));
        } else {
            acc = product(acc, [&](int s) {
                const int t = 2 * s + hi;
                return Km[t * KP + it * 32 + l32] * Wc[max(nc - 1 - t, 0)];      // (k is zero past the end)
            }, across(Vm, VP, ct * 32));
        }
        check(acc);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int kt = it * 2 + (q >> 1), g = (q & 1) * 2 + hi, cb = ct * 2 + (l32 >> 4);
            *reinterpret_cast<float4*>(unit + U::S + ((cb * (DK / 16) + kt) * 64 + g * 16 + (l32 & 15)) * 4) =
                make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
        }
    }
    if (DELTA) {
        // M transposed (rows: the channel it is summed over, columns: the channel it goes to)
        for (int m = wave; m < TK * TK; m += 4) {
            const int jt = m / TK, it = m % TK;
            const float wc = Wc[it * 32 + l32];
            f32x16_t acc = minus(product(f32x16_t{}, across(Xm, XP, jt * 32),
                                         [&](int s) { return Bm[(2 * s + hi) * KP + it * 32 + l32] * wc; }));
#pragma unroll
            for (int e = 0; e < 16; ++e)
                if (jt == it && 8 * (e >> 2) + 4 * hi + (e & 3) == l32) acc[e] += wc;
            check(acc);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int kt = jt * 2 + (q >> 1), g = (q & 1) * 2 + hi, rt = it * 2 + (l32 >> 4);
                *reinterpret_cast<float4*>(unit + U::M + ((rt * (DK / 16) + kt) * 64 + g * 16 + (l32 & 15)) * 4) =
                    make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
            }
        }
    }
    const int any = __syncthreads_or(bad);
    if (tid == 0) reinterpret_cast<int*>(unit)[U::BAD] = any;
}

// The state through the segment's chunks, 16 of its columns a block.  A wave owns 32 rows (two tiles of 16); with
// v_mfma_f32_16x16x4_f32 a result (row 4 g + i, column l % 16 in element i of lane 16 g + l % 16) is the operand of
// the next product as it lies, for the four k values {16 a + 4 g + i}: the operators are stored for that order.  The
// waves hand their rows to each other through LDS.
template <int DK, int DV, bool DELTA>
__global__ __launch_bounds__(DK * 2) void chunk_states_kernel(const ChunkArgs a) {
    constexpr int NW = DK / 32, NA = DK / 16;
    using U = Unit<DK, DV, DELTA>;
    const int b = blockIdx.z, h = blockIdx.y, cb = blockIdx.x;
    const int t_lo = a.cu_q[b], n = a.cu_q[b + 1] - t_lo;
    if (n < a.min_tokens || a.c0 * C >= n) return;
    int* const from = a.from + ((size_t)b * a.H + h) * (DV / 16) + cb;       // (this block's own, the same in all of a head's)
    if (a.c0 > 0 && *from < a.c0 * C) return;          // the walk takes the row over before this segment
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, g = lane >> 4;
    const int all = min(a.seg, (n + C - 1) / C - a.c0);          // at most 64
    const float* units = a.ws + ((size_t)b * a.seg * a.H + h) * U::SIZE;
    const unsigned long long bads = __ballot(lane < all && reinterpret_cast<const int*>(units + (size_t)lane * a.H * U::SIZE)[U::BAD] != 0);
    const int chunks = bads ? __ffsll(bads) - 1 : all;
    if (threadIdx.x == 0) *from = (a.c0 + chunks) * C;
    __shared__ __align__(16) f32x4_t St[2][NA][64];
    float* Sg = a.state + ((size_t)a.slots[b] * a.H + h) * (size_t)DK * DV + cb * 16 + col;
    const bool fresh = a.c0 == 0 && a.q_start[b] == 0;
    f32x4_t S[2];
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) S[q][i] = fresh ? 0.f : Sg[(size_t)((wave * 2 + q) * 16 + 4 * g + i) * DV];
    struct Ops { f32x4_t m[DELTA ? 2 : 1][DELTA ? NA : 1], r[NA], add[2], o; };
    const bool outputs = wave < 2;               // two tiles of 16 tokens
    const float d = DELTA ? 0.f : a.decay[h];
    const float d_chunk = DELTA ? 0.f : power(d, C);
    auto ask = [&](int c, Ops& x) {
        const f32x4_t* unit = reinterpret_cast<const f32x4_t*>(units + (size_t)c * a.H * U::SIZE);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            x.add[q] = unit[U::S / 4 + (cb * NA + wave * 2 + q) * 64 + lane];
            if (DELTA) {
#pragma unroll
                for (int k = 0; k < NA; ++k) x.m[q][k] = unit[U::M / 4 + ((wave * 2 + q) * NA + k) * 64 + lane];
            }
        }
        if (outputs) {
#pragma unroll
            for (int k = 0; k < NA; ++k) x.r[k] = unit[U::R / 4 + (wave * NA + k) * 64 + lane];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = (a.c0 + c) * C + wave * 16 + 4 * g + i;
                x.o[i] = t < n ? a.out[(size_t)(t_lo + t) * a.out_stride + h * DV + cb * 16 + col] : 0.f;
            }
        }
    };
    auto step = [&](int c, Ops& x) {
#pragma unroll
        for (int q = 0; q < 2; ++q) St[c & 1][wave * 2 + q][lane] = S[q];
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // LDS only: the next chunk's loads stay under way
        const float dc = DELTA ? 0.f : ((a.c0 + c + 1) * C <= n ? d_chunk : power(d, n - (a.c0 + c) * C));
        constexpr int CH = 4;                                                // chains of sums, as in product
        f32x4_t next[2][CH] = {}, o[CH] = {};
#pragma unroll
        for (int k = 0; k < NA; ++k) {
            const f32x4_t s = St[c & 1][k][lane];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (DELTA) {
                    next[0][i % CH] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.m[0][k][i], s[i], next[0][i % CH], 0, 0, 0);
                    next[1][i % CH] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.m[1][k][i], s[i], next[1][i % CH], 0, 0, 0);
                }
                if (outputs) o[i % CH] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.r[k][i], s[i], o[i % CH], 0, 0, 0);
            }
        }
        const auto whole = [](const f32x4_t (&p)[CH]) { return (p[0] + p[1]) + (p[2] + p[3]); };
        if (outputs) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = (a.c0 + c) * C + wave * 16 + 4 * g + i;
                if (t < n) a.out[(size_t)(t_lo + t) * a.out_stride + h * DV + cb * 16 + col] = x.o[i] + whole(o)[i];
            }
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            if (DELTA) {
                S[q] = x.add[q] + whole(next[q]);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) S[q][i] = fmaf(dc, S[q][i], x.add[q][i]);
            }
        }
    };
    static_assert(NW >= 2, "two waves make the outputs");
    Ops x0, x1;
    if (chunks > 0) ask(0, x0);
    for (int c = 0; c < chunks; c += 2) {
        if (c + 1 < chunks) ask(c + 1, x1);
        step(c, x0);
        if (c + 1 < chunks) {
            if (c + 2 < chunks) ask(c + 2, x0);
            step(c + 1, x1);
        }
    }
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) Sg[(size_t)((wave * 2 + q) * 16 + 4 * g + i) * DV] = S[q][i];
}

template <int DK, int DV, bool DELTA>
int launch_chunks(ChunkArgs a, int num_rows, int max_tokens, hipStream_t stream) {
    constexpr int KP = DK + 4, VP = DV + 4;
    constexpr size_t lds = sizeof(float) * (C * (2 * KP + VP + CP) + (DK > C + 4 ? DK : C + 4)
                                            + (DELTA ? C * (2 * KP + 3 * CP + DK + DV + 4) : 0));
    static_assert(lds <= 160 * 1024, "more LDS than a compute unit has");
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
        operators<<<dim3(min(a.seg, chunks - a.c0), a.H, num_rows), 256, lds, stream>>>(a);
        chunk_states_kernel<DK, DV, DELTA><<<dim3(DV / 16, a.H, num_rows), DK * 2, 0, stream>>>(a);
    }
    return 0;
}

// chunks of every row that one pass takes: the workspace holds some 64 chunks of all heads
int segment(int num_rows, int max_tokens) {
    const int chunks = (max_tokens + C - 1) / C, most = num_rows < 64 ? 64 / num_rows : 1;
    return chunks < most ? chunks : most;
}

}  // namespace

// Whether ri_linear_scan_chunks takes heads of this size (delta: with decays of at least exp(-decay_c)).
extern "C" int ri_linear_scan_chunks_supported(int delta, int dk, int dv, float decay_c) {
    if (delta && !(decay_c >= 0.f && decay_c * C <= 60.f)) return 0;      // W_C >= 1e-26
    return (dk == 64 || dk == 128) && dv == dk;
}

static size_t unit_floats(int delta, int num_rows, int max_tokens, int H, int dk, int dv) {
    return (size_t)num_rows * segment(num_rows, max_tokens) * H * ((size_t)C * dk + (size_t)dk * dv + (delta ? (size_t)dk * dk : 0) + 4);
}

// Floats of workspace for steps of up to num_rows rows of at most max_tokens tokens.
extern "C" size_t ri_linear_scan_chunks_workspace(int delta, int num_rows, int max_tokens, int H, int dk, int dv) {
    return unit_floats(delta, num_rows, max_tokens, H, dk, dv) + (size_t)num_rows * H * (dv / 16);
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
// does the others, and what the chunks leave to it.  bfloat16 projections.
extern "C" int ri_linear_scan_chunks(
        const void* r, int r_stride, const void* k, int k_stride, const void* v, int v_stride,
        const void* wl, int wl_stride, const void* al, int al_stride,
        const float* w0, const float* ab, const float* decay, int delta, int silu_in,
        float unit_eps, float decay_c, float* state, int num_slots, float* out, int out_stride,
        const int* cu_q, const int* q_start, const int* slots, int num_rows, int T,
        int H, int dk, int dv, const float* rot_cos, const float* rot_sin, int rot, int rot_rows, int max_position,
        float k_scale, int min_tokens, int max_tokens, float* ws, size_t ws_floats, hipStream_t stream) {
    RI_REQUIRE(H > 0 && ri_linear_scan_chunks_supported(delta, dk, dv, decay_c), "ri_linear_scan_chunks: does not take H=%d dk=%d dv=%d decay_c=%g", H, dk, dv, (double)decay_c);
    RI_REQUIRE(num_rows >= 0 && T >= 0 && num_slots > 0 && min_tokens > 1, "ri_linear_scan_chunks: bad counts");
    RI_REQUIRE(r_stride >= H * dk && k_stride >= H * dk && v_stride >= H * dv && out_stride >= H * dv, "ri_linear_scan_chunks: row strides too small");
    if (num_rows == 0 || T == 0 || max_tokens <= 0) return 0;
    RI_REQUIRE(r && k && v && state && out && cu_q && q_start && slots && ws, "ri_linear_scan_chunks: null pointer");
    RI_REQUIRE(H <= 65535 && num_rows <= 65535, "ri_linear_scan_chunks: too many heads or rows for the grid");
    RI_REQUIRE((uintptr_t)ws % 16 == 0 && ws_floats >= ri_linear_scan_chunks_workspace(delta, num_rows, max_tokens, H, dk, dv), "ri_linear_scan_chunks: the workspace is too small");
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
    a.ws = ws; a.c0 = 0; a.seg = segment(num_rows, max_tokens);
    a.from = reinterpret_cast<int*>(ws + unit_floats(delta, num_rows, max_tokens, H, dk, dv));
    int rc;
    if (dk == 64) rc = delta ? launch_chunks<64, 64, true>(a, num_rows, max_tokens, stream) : launch_chunks<64, 64, false>(a, num_rows, max_tokens, stream);
    else rc = delta ? launch_chunks<128, 128, true>(a, num_rows, max_tokens, stream) : launch_chunks<128, 128, false>(a, num_rows, max_tokens, stream);
    if (rc) return rc;
    RI_LAUNCHED("ri_linear_scan_chunks");
    return ri_linear_scan(r, r_stride, k, k_stride, v, v_stride, wl, wl_stride, al, al_stride, RI_BF16, w0, ab, decay, delta, silu_in,
                          unit_eps, decay_c, state, num_slots, out, out_stride, cu_q, q_start, slots, num_rows, T, H, dk, dv,
                          rot_cos, rot_sin, rot, rot_rows, max_position, k_scale, min_tokens - 1, a.from, dv / 16, stream);
}
