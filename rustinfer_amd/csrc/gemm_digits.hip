// gemm_digits: C[M, N] = A[M, K] . W[N, K]^T of 32-bit operands on the 8-bit integer matrix instruction, for the 32-bit path's prompts, each
// result as near to the product of the 32-bit values as a 64-bit sum of them (gemm_f32.hip) leaves it.
//
// Each row is brought to whole numbers below its own largest value: x = q 2^(e - 47), e the least exponent that holds the row's largest magnitude,
// q to six digits of eight bits, base 256, from -128 to 127; rows of W to five (2^(e - 39)).  Of the 30 products of digits the 20 whose digits
// (counted from the first) add up to five at most are summed, each in 32-bit integers that cannot overflow (K <= 26,000), and put together exactly: the
// one rounding on the way is that of 53 bits.  What that leaves out of a result is bounded by what it is, not by the largest values: with N_i the 2-norm
// of a row's digit i, T_j that of a row of W from digit j on (in units of digit j), n a row's norm and c that of what was cut off below its last digit,
//     |error| <= 2^-62 (N_2 T_4 + N_3 T_3 + N_4 T_2 + N_5 T_1) + c_x n_w + n_x c_w        (in units of both rows' exponents)
// by the inequality of Cauchy and Schwarz, and a result smaller than 2^27 times that is computed again from the 32-bit values in 64-bit sums.  So every
// result is within half a unit of its last place and 2^-27 of itself, or a 64-bit sum.  What is lost in fact is a twelfth to a fortieth of the bound.  How many are computed again: of normal rows
// against normal weights 0.03 % (K = 2048) and 0.07 % (8192), of a gated activation 0.1 and 0.2 %, with a value of 2^16 standard deviations in each row 0.4 and 4 %.  Their places are
// noted a row at a time, N / 16 of them at most; a wave does such a result in 64-bit FMAs.  A row that has more goes to the kernel of 64-bit
// sums whole, with the others like it, and so do rows that hold an infinity or a NaN, and rows most of whose values are cut off (these two without being
// multiplied first where all 64 rows of a block are such).  A weight with such a row gets no digits.
//
// Digits lie as the matrix instruction takes them: [rows / 32][K / 32][digits][64 lanes][16 bytes], lane 32 h + r holding k = 16 h .. 16 h + 15 of
// row r, the first digit first.  A block of eight waves makes 64 x 128 results: a stage of 32 values of K (32 KiB) goes straight into LDS while
// the stage before is multiplied; two such blocks fit a unit.  What bounds it: the instruction at the clock that the card's power leaves it (a
// loop of it alone reaches 4.7 POP/s on zeros and 3.4 on random digits; this kernel 2.4).  Measured, us, 64-bit sums / this with all that goes with it:
// 600 rows of 16384 x 2048 724 / 362, 3072 x 2048 128 / 82, 2048 x 2048 95 / 71, 2048 x 8192 (a gated activation) 350 / 222; 194 rows 250 / 141
// (16384 x 2048), 135 / 91 (2048 x 8192); 89 rows 113 / 81, 85 / 59.  (Five digits for both and 15 products, without the bound: 264 us for the
// first, and results that were off by as much as their size where large values of the one row met small ones of the other.)  600 rows of which 1, 60, 600
// have no digits: 16384 x 2048 462, 455, 765, 2048 x 8192 285, 284, 369, 2048 x 2048 90, 91, 112; all with a value of 2^12 standard deviations: 380, 330, 78 (2048 x 8192
// with N / 32 places a row, so that 61 rows were done whole: 385).
#include "common.h"
#include <float.h>
#include <limits.h>

typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x16_t __attribute__((ext_vector_type(16)));

extern "C" void ri_gemm_f32_tile(int M, int N, int* rows, int* columns);      // gemm_f32.hip
extern "C" int ri_gemm_f32_listed(const float* A, int lda, const float* W, int ldw, float* C, int ldc, int M, int N, int K,
                                  const int* list, hipStream_t stream);      // gemm_f32.hip

namespace {

constexpr int DA = 6, DW = 5, SUMS = 6;                       // digits of A and of W; sums of products by the sum of the digits' numbers
constexpr int PIECE_A = DA * 1024, PIECE_W = DW * 1024;       // bytes of 32 rows by 32 values of K
constexpr int MAX_K = 26000;                                  // 5 products of at most 2^14 a value of K in 32-bit sums
constexpr float AGAIN = 1.01f * 134217728.f;                  // 2^27, and what the roundings of the bound itself may take

// What is known of a row.  A: the norms N_2 to N_5, then c and n; W: T_4, T_3, T_2, T_1, then n and c, so that the bound is the sum of six products in order.
// In units in which the products are 2^-54 of the exponents' (digit 5 of a product): see bound().  part[0] = infinity: a row without digits.
struct RowOf {
    float part[6];
    int e, unused;
};

// s_waitcnt: at most n loads under way, and nothing asked of LDS: a stage is written over behind the barrier only when what was read of it has arrived
constexpr int loads_imm(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4); }

__device__ __forceinline__ float bound(const float (&x)[6], const float (&w)[6]) {
    float b = x[0] * w[0];
#pragma unroll
    for (int i = 1; i < 6; ++i) b = fmaf(x[i], w[i], b);
    return b * AGAIN;
}

__device__ __forceinline__ float to_float(double v, int ea, int ew) {
    return (float)(v * __longlong_as_double((long long)(1023 + ea + ew - 54) << 52));
}

// What is to be computed again, in one buffer of integers: the rows to be done whole, their number first, the count of each row's noted results, then
// the columns of those, `cap` places a row.  A count that has passed `cap` is that of a row to be done whole; whoever takes it past puts the row on the list.
struct Again {
    int* rows;               // [1 + M]
    int* counts;             // [M]
    int* columns;            // [M][cap]
    int cap;
    __host__ __device__ Again(int* buffer, int M, int N) : rows(buffer), counts(buffer + 1 + M), columns(buffer + 1 + 2 * (size_t)M), cap(N / 16) {}
    // places for `many` results of row m, from the returned one on
    __device__ __forceinline__ int note(int m, int many) const {
        const int old = atomicAdd(counts + m, many);
        if (old <= cap && old + many > cap) rows[1 + atomicAdd(rows, 1)] = m;
        return old;
    }
};

// The digits of rows and what is known of them.  A block a row (rows of a last tile beyond the end are zeros), sixteen values a thread and turn,
// read for the largest, then for the digits, the first turn's kept.  Four rows that follow each other run on one XCD, so that the 16 bytes a row
// leaves of each line meet in one L2.
template <int D>
__global__ __launch_bounds__(512, 4) void digits_split_kernel(const float* __restrict__ X, int ld, int rows, int K, uint8_t* __restrict__ planes,
                                                           RowOf* __restrict__ known, Again again) {
    constexpr int BITS = 8 * D - 1, PIECE = D * 1024, FIRST = D - 4;      // FIRST: of the digits whose norms are kept
    __shared__ uint32_t largest[8];
    __shared__ int above[8];
    __shared__ uint32_t squares[8][4];
    __shared__ float norms[8][2];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, waves = blockDim.x >> 6;
    const int b = blockIdx.x, row = (b >> 5) * 32 + (b & 7) * 4 + ((b >> 3) & 3);
    const bool in = row < rows;
    const float* x = X + (size_t)(in ? row : 0) * ld;
    uint32_t most = 0;
    const int first = threadIdx.x * 16;
    float4 kept[4] = {};                                         // of the first turn, the only one up to 8,192 values
    auto look = [&](const float4& v) {
        most = max(most, max(max(__float_as_uint(v.x) & 0x7fffffffu, __float_as_uint(v.y) & 0x7fffffffu),
                             max(__float_as_uint(v.z) & 0x7fffffffu, __float_as_uint(v.w) & 0x7fffffffu)));
    };
    if (in && first < K)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            kept[q] = *reinterpret_cast<const float4*>(x + first + 4 * q);
            look(kept[q]);
        }
    if (in)
        for (int k = first + blockDim.x * 16; k < K; k += blockDim.x * 16)
#pragma unroll
            for (int q = 0; q < 4; ++q) look(*reinterpret_cast<const float4*>(x + k + 4 * q));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) most = max(most, (uint32_t)__shfl_xor((int)most, o, 64));
    if (lane == 0) largest[wave] = most;
    __syncthreads();
    for (int i = 0; i < waves; ++i) most = max(most, largest[i]);
    const bool finite = most < 0x7f800000u;
    int e = 0;
    if (most && finite) {
        // the largest and a 128th more are below 2^e: its first digit, with what the others' signs carry into it, is at most 127
        const double up = (double)__uint_as_float(most) * (1.0 + 1.0 / 127.0);
        e = (int)(__double_as_longlong(up) >> 52) - 1022;
    }
    const double scale = __longlong_as_double((long long)(1023 + BITS - e) << 52);
    uint8_t* out = planes + (size_t)(row >> 5) * (K / 32) * PIECE + (row & 31) * 16;
    // below `small` a value loses bits (W: or nearly so)
    const float small = __uint_as_float(most) * (D == 6 ? 0x1p-24f : 0x1p-13f);
    int balance = 0;
    uint32_t sq[4] = {};
    float n2 = 0.f, c2 = 0.f;
    for (int k = first; k < K; k += blockDim.x * 16) {
        uint32_t d[D][4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float4 f = make_float4(0.f, 0.f, 0.f, 0.f);
            if (in && finite) f = k == first ? kept[q] : *reinterpret_cast<const float4*>(x + k + 4 * q);
            const float v[4] = {f.x, f.y, f.z, f.w};
            uint32_t lo[4], hi[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                balance += v[j] == 0.f ? 0 : fabsf(v[j]) >= small ? 1 : -1;
                const double t = (double)v[j] * scale, whole = rint(t);
                const float cut = (float)(t - whole), near = (float)whole;
                c2 = fmaf(cut, cut, c2);
                n2 = fmaf(near, near, n2);
                const long long n = (long long)whole + (D == 6 ? 0x8080808080ll : 0x80808080ll);
                lo[j] = (uint32_t)n ^ 0x80808080u;                               // the last four digits, signed bytes, the last one first
                hi[j] = (uint32_t)(n >> 32) ^ (D == 6 ? 0x80u : 0u);             // and the first (two)
            }
            // bytes of four values to four values a digit: two digits of two values each, then one of four
            const uint32_t p01 = __builtin_amdgcn_perm(lo[1], lo[0], 0x05010400u), q01 = __builtin_amdgcn_perm(lo[1], lo[0], 0x07030602u);
            const uint32_t p23 = __builtin_amdgcn_perm(lo[3], lo[2], 0x05010400u), q23 = __builtin_amdgcn_perm(lo[3], lo[2], 0x07030602u);
            const uint32_t r01 = __builtin_amdgcn_perm(hi[1], hi[0], 0x05010400u), r23 = __builtin_amdgcn_perm(hi[3], hi[2], 0x05010400u);
            d[D - 1][q] = __builtin_amdgcn_perm(p23, p01, 0x05040100u);
            d[D - 2][q] = __builtin_amdgcn_perm(p23, p01, 0x07060302u);
            d[D - 3][q] = __builtin_amdgcn_perm(q23, q01, 0x05040100u);
            d[D - 4][q] = __builtin_amdgcn_perm(q23, q01, 0x07060302u);
            d[D - 5][q] = __builtin_amdgcn_perm(r23, r01, 0x05040100u);
            if (D == 6) d[0][q] = __builtin_amdgcn_perm(r23, r01, 0x07060302u);
#pragma unroll
            for (int i = 0; i < 4; ++i) sq[i] = (uint32_t)__builtin_amdgcn_sdot4((int)d[FIRST + i][q], (int)d[FIRST + i][q], (int)sq[i], false);
        }
        uint8_t* o = out + (size_t)(k >> 5) * PIECE + ((k >> 4) & 1) * 512;
#pragma unroll
        for (int i = 0; i < D; ++i) *reinterpret_cast<uint4*>(o + i * 1024) = make_uint4(d[i][0], d[i][1], d[i][2], d[i][3]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        balance += __shfl_xor(balance, o, 64);
        n2 += __shfl_xor(n2, o, 64);
        c2 += __shfl_xor(c2, o, 64);
#pragma unroll
        for (int i = 0; i < 4; ++i) sq[i] += (uint32_t)__shfl_xor((int)sq[i], o, 64);
    }
    if (lane == 0) {
        above[wave] = balance;
        norms[wave][0] = n2;
        norms[wave][1] = c2;
#pragma unroll
        for (int i = 0; i < 4; ++i) squares[wave][i] = sq[i];
    }
    __syncthreads();
    if (threadIdx.x) return;
    for (int i = 1; i < waves; ++i) {
        balance += above[i];
        n2 += norms[i][0];
        c2 += norms[i][1];
#pragma unroll
        for (int j = 0; j < 4; ++j) sq[j] += squares[i][j];
    }
    const bool has = finite && balance >= 0;
    // n and c by 2^27 each, so that their products are in units of 2^-54; n with what was cut off, as the bound has the whole row once
    const float unit = D == 6 ? 0x1p-20f : 0x1p-12f, c = sqrtf(c2) * unit, n = sqrtf(n2) * unit + c;
    RowOf k;
    if (D == 6) {
#pragma unroll
        for (int i = 0; i < 4; ++i) k.part[i] = sqrtf((float)sq[i]);
        k.part[4] = c;
        k.part[5] = n;
    } else {
        // T_j = N_j + T_(j + 1) / 256; a unit of digit 6 of a product is 2^-8 of one of digit 5
        float t = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            t = sqrtf((float)sq[3 - i]) + t * 0x1p-8f;
            k.part[i] = t * 0x1p-8f;
        }
        k.part[4] = n;
        k.part[5] = c + n * 0x1p-48f;                            // and the roundings of up to 16 slices' 53 bits
    }
    if (!has) k.part[0] = INFINITY;
    k.e = e;
    k.unused = 0;
    known[row] = k;
    if (again.rows && in) {
        again.counts[row] = has ? 0 : again.cap;                 // one result more, and the row is done whole
        if (row == 0) again.rows[0] = 0;
    }
}

// 2 x 4 waves of 32 x 32 results.  blockIdx.y: the slice of K, `part` chunks of 32 values; with several, sums
// [parts][M][N] are left in P for digits_sum_kernel, else the results in C.
__global__ __launch_bounds__(512, 4) void gemm_digits_kernel(
        const uint8_t* __restrict__ A, const RowOf* __restrict__ ka, const uint8_t* __restrict__ W, const RowOf* __restrict__ kw,
        float* __restrict__ C, int ldc, double* __restrict__ P, Again again, int M, int N, int K, int part, int mblocks, int nblocks) {
    constexpr int WM = 2, WN = 4, WAVES = WM * WN, FRAGS = WM * DA + WN * DW, PER = FRAGS / WAVES, STAGE = FRAGS * 1024;
    static_assert(FRAGS % WAVES == 0, "a wave brings in as many kilobytes of a stage as the others");
    __shared__ __align__(16) uint8_t lds[2 * STAGE];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave % WM, wn = wave / WM;
    // the row blocks of one block of columns run on one XCD (consecutive block ids go around the eight of them)
    const int id = (int)blockIdx.x, turn = id >> 3;
    const int nb = (turn / mblocks) * 8 + (id & 7), mb = turn % mblocks;
    if (nb >= nblocks) return;
    const int mtiles = (M + 31) / 32, ntiles = N / 32, chunks = K / 32;
    // tiles beyond the end are read (clamped), never stored
    const uint8_t* from[PER];
    int step[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int f = wave * PER + i;
        if (f < WM * DA) {
            from[i] = A + (size_t)min(mb * WM + f / DA, mtiles - 1) * chunks * PIECE_A + f % DA * 1024;
            step[i] = PIECE_A;
        } else {
            from[i] = W + (size_t)min(nb * WN + (f - WM * DA) / DW, ntiles - 1) * chunks * PIECE_W + (f - WM * DA) % DW * 1024;
            step[i] = PIECE_W;
        }
    }
    auto fetch = [&](int c, int at) {
#pragma unroll
        for (int i = 0; i < PER; ++i)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(from[i] + (size_t)c * step[i] + lane * 16),
                (__attribute__((address_space(3))) void*)(lds + at + (wave * PER + i) * 1024), 16, 0, 0);
    };
    // acc[s]: the products of digits i and j with i + j = s
    i32x16_t acc[SUMS] = {};
    const int c0 = blockIdx.y * part, c1 = min(chunks, c0 + part);
    // rows without digits are put on the list by the first block of columns and left alone by all; a block of nothing else ends here (the same answer in every wave)
    const bool row = mb * 64 + lane < M, has = row && ka[min(mb * 64 + lane, M - 1)].part[0] != INFINITY;
    if (nb == 0 && blockIdx.y == 0 && wave == 0 && row && !has) again.note(mb * 64 + lane, 1);
    if (__ballot(has) == 0) return;
    if (c0 < c1) fetch(c0, 0);
    int at = 0;
    for (int c = c0; c < c1; ++c) {
        __builtin_amdgcn_s_waitcnt(loads_imm(0));                // this wave's part of the stage has arrived, and behind the barrier everyone's;
        __builtin_amdgcn_s_barrier();                            // all have read the other one
        asm volatile("" ::: "memory");
        if (c + 1 < c1) fetch(c + 1, STAGE - at);
        const i32x4_t* la = reinterpret_cast<const i32x4_t*>(lds + at + wm * PIECE_A) + lane;
        const i32x4_t* lw = reinterpret_cast<const i32x4_t*>(lds + at + WM * PIECE_A + wn * PIECE_W) + lane;
        // three digits of A against all of W's, then the other three: registers for all of both would not be there beside the sums
#pragma unroll
        for (int h = 0; h < DA; h += 3) {
            i32x4_t a[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) a[i] = la[(h + i) * 64];
#pragma unroll
            for (int j = 0; j < DW && h + j < SUMS; ++j) {
                const i32x4_t b = lw[j * 64];
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    if (h + i + j < SUMS) acc[h + i + j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[i], b, acc[h + i + j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        at = STAGE - at;
    }
    // result (row 8 (i / 4) + 4 (lane / 32) + i % 4, column lane % 32) of a tile lies in element i
    const int n = (nb * WN + wn) * 32 + (lane & 31), m0 = (mb * WM + wm) * 32;
    RowOf* rows = reinterpret_cast<RowOf*>(lds);                 // what is known of the block's rows
    __syncthreads();
    if (threadIdx.x < 128) reinterpret_cast<float4*>(rows)[threadIdx.x] = reinterpret_cast<const float4*>(ka + min(mb * 64 + (int)threadIdx.x / 2, M - 1))[threadIdx.x & 1];
    __syncthreads();
    if ((nb * WN + wn) * 32 >= N || m0 >= M) return;
    const RowOf w = kw[n];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int m = m0 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
        // both parts are whole numbers below 2^53: one rounding
        const long long high = (((long long)acc[0][i] * 256 + acc[1][i]) * 256 + acc[2][i]) * 256 + acc[3][i], low = (long long)acc[4][i] * 256 + acc[5][i];
        const double v = fma((double)high, 65536.0, (double)low);
        if (P) {
            if (m < M) P[((size_t)blockIdx.y * M + m) * N + n] = v;
            continue;
        }
        const RowOf x = rows[m - mb * 64];
        bool redo = false;
        if (m < M && x.part[0] != INFINITY) {
            redo = !(fabsf((float)v) >= bound(x.part, w.part));
            C[(size_t)m * ldc + n] = to_float(v, x.e, w.e);
        }
        const uint64_t all = __ballot(redo);
        if (all == 0) continue;
        const uint32_t mine = lane < 32 ? (uint32_t)all : (uint32_t)(all >> 32);      // of the lanes with this row
        int old = 0;
        if ((lane & 31) == 0 && mine) old = again.note(m, __popc(mine));
        old = __shfl(old, lane & 32, 64) + __popc(mine & ((1u << (lane & 31)) - 1));
        if (redo && old < again.cap) again.columns[(size_t)m * again.cap + old] = n;
    }
}

// The slices' sums, added up and rounded once: a block 256 columns of a row.
__global__ __launch_bounds__(256) void digits_sum_kernel(const double* __restrict__ P, int parts, const RowOf* __restrict__ ka, const RowOf* __restrict__ kw,
                                                         float* __restrict__ C, int ldc, Again again, int M, int N) {
    const int m = blockIdx.y, n = blockIdx.x * 256 + threadIdx.x, lane = threadIdx.x & 63;
    const RowOf x = ka[m];
    if (x.part[0] == INFINITY) return;
    bool redo = false;
    if (n < N) {
        const RowOf w = kw[n];
        double v = 0.0;
        for (int p = 0; p < parts; ++p) v += P[((size_t)p * M + m) * N + n];
        redo = !(fabsf((float)v) >= bound(x.part, w.part));
        C[(size_t)m * ldc + n] = to_float(v, x.e, w.e);
    }
    const uint64_t all = __ballot(redo);
    if (all == 0) return;
    int old = 0;
    if (lane == 0) old = again.note(m, __popcll(all));
    old = __shfl(old, 0, 64) + __popcll(all & ((1ull << lane) - 1));
    if (redo && old < again.cap) again.columns[(size_t)m * again.cap + old] = n;
}

// The results that were noted, a wave each: a 64-bit sum, the lanes' shares in the order of K.  Bound by the rows of W, most of which are read for some result:
// 3,000 results of 600 rows of 2048 x 8192 24 us, 67 MB of W among what is read (a block each 23); 2,700 of 16384 x 2048 10.
__global__ __launch_bounds__(256) void digits_again_kernel(const float* __restrict__ X, int ldx, const float* __restrict__ W, int ldw, float* __restrict__ C, int ldc,
                                                           Again again, int K) {
    const int m = blockIdx.x, lane = threadIdx.x & 63, count = again.counts[m];
    if (count > again.cap) return;
    for (int i = (int)(blockIdx.y * 4 + (threadIdx.x >> 6)); i < count; i += gridDim.y * 4) {
        const int n = again.columns[(size_t)m * again.cap + i];
        const float *x = X + (size_t)m * ldx, *w = W + (size_t)n * ldw;
        double v = 0.0;
#pragma unroll 8
        for (int k = lane * 4; k < K; k += 256) {
            const float4 a = *reinterpret_cast<const float4*>(x + k), b = *reinterpret_cast<const float4*>(w + k);
            v = fma((double)a.x, (double)b.x, v);
            v = fma((double)a.y, (double)b.y, v);
            v = fma((double)a.z, (double)b.z, v);
            v = fma((double)a.w, (double)b.w, v);
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        if (lane == 0) C[(size_t)m * ldc + n] = (float)v;
    }
}

}  // namespace

// Bytes of the digits of `rows` rows of K values (whole tiles of 32 rows), six digits a value for the rows of a product and five for its weight.
extern "C" long long ri_digits_bytes(int rows, int K, int digits) { return (long long)((rows + 31) / 32) * (K / 32) * digits * 1024; }

extern "C" int ri_digits_max_k() { return MAX_K; }

// Digits of X[rows, K] and what is known of each row (eight 32-bit words, rows up to whole tiles of 32; a row without digits has an infinity in the first).
// For the rows of a product of N columns, `again`: the buffer of (1 + 2 rows + rows (N / 16)) integers that ri_gemm_digits takes.
extern "C" int ri_digits_split(const float* X, int ld, int rows, int K, int digits, void* planes, void* known, int* again, int N, hipStream_t stream) {
    RI_REQUIRE(rows >= 1 && K >= 32 && K % 32 == 0 && K <= MAX_K, "ri_digits_split: needs K %% 32 == 0 and at most %d (rows=%d K=%d)", MAX_K, rows, K);
    RI_REQUIRE(digits == DA || digits == DW, "ri_digits_split: %d digits, not %d or %d", digits, DA, DW);
    RI_REQUIRE(ld >= K && ld % 4 == 0, "ri_digits_split: bad leading dimension");
    RI_REQUIRE(X && planes && known && (uintptr_t)X % 16 == 0 && (uintptr_t)planes % 16 == 0 && (uintptr_t)known % 16 == 0, "ri_digits_split: null or unaligned pointer");
    RI_REQUIRE(rows <= (1 << 22) && N >= 0, "ri_digits_split: rows=%d exceed the grid limit", rows);
    RI_REQUIRE((digits == DA) == (again != nullptr), "ri_digits_split: a product's rows go with the list of what is computed again, a weight's do not");
    const int threads = min(512, (K / 16 + 63) / 64 * 64), blocks = (rows + 31) / 32 * 32;
    Again list(again, rows, N);
    if (digits == DA) digits_split_kernel<DA><<<blocks, threads, 0, stream>>>(X, ld, rows, K, (uint8_t*)planes, (RowOf*)known, list);
    else digits_split_kernel<DW><<<blocks, threads, 0, stream>>>(X, ld, rows, K, (uint8_t*)planes, (RowOf*)known, list);
    RI_LAUNCHED("ri_digits_split");
    return 0;
}

// C[M, N] from the digits of A (of the rows X, ldx) and of W (w32: its 32-bit values), and what is known of both.  parts > 1: slices of K, sums [parts][M][N].
extern "C" int ri_gemm_digits(const void* A, const void* ka, const float* X, int ldx, const void* W, const void* kw,
                              const float* w32, int ldw, float* C, int ldc, double* sums, int parts, int* again,
                              int M, int N, int K, hipStream_t stream) {
    RI_REQUIRE(M >= 1 && N >= 32 && N % 32 == 0 && K >= 32 && K % 32 == 0 && K <= MAX_K,
               "ri_gemm_digits: needs N and K in multiples of 32, K at most %d (M=%d N=%d K=%d)", MAX_K, M, N, K);
    RI_REQUIRE(A && ka && X && W && kw && w32 && C && again && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0 && (uintptr_t)X % 16 == 0
               && (uintptr_t)w32 % 16 == 0 && (uintptr_t)ka % 16 == 0 && (uintptr_t)kw % 16 == 0, "ri_gemm_digits: null or unaligned pointer");
    RI_REQUIRE(ldx >= K && ldx % 4 == 0 && ldw >= K && ldw % 4 == 0 && ldc >= N && ldx <= (1 << 24) && ldw <= (1 << 24), "ri_gemm_digits: bad leading dimensions");
    RI_REQUIRE(parts >= 1 && parts <= 16 && (parts == 1 || sums), "ri_gemm_digits: parts=%d", parts);
    const int mblocks = (M + 63) / 64, nblocks = (N + 127) / 128, chunks = K / 32;
    const long long blocks = (long long)((nblocks + 7) / 8 * 8) * mblocks;
    RI_REQUIRE(blocks * parts < (1 << 22) && M <= 65535, "ri_gemm_digits: M=%d N=%d exceed the grid limit", M, N);
    const Again list(again, M, N);
    gemm_digits_kernel<<<dim3((unsigned)blocks, parts), 512, 0, stream>>>((const uint8_t*)A, (const RowOf*)ka, (const uint8_t*)W, (const RowOf*)kw, C, ldc,
        parts > 1 ? sums : nullptr, list, M, N, K, (chunks + parts - 1) / parts, mblocks, nblocks);
    RI_LAUNCHED("ri_gemm_digits");
    if (parts > 1) {
        digits_sum_kernel<<<dim3((N + 255) / 256, M), 256, 0, stream>>>(sums, parts, (const RowOf*)ka, (const RowOf*)kw, C, ldc, list, M, N);
        RI_LAUNCHED("ri_gemm_digits");
    }
    // a row's places by several blocks where the rows are few
    const int across = max(1, min((list.cap + 3) / 4, (1024 + M - 1) / M));
    digits_again_kernel<<<dim3(M, across), 256, 0, stream>>>(X, ldx, w32, ldw, C, ldc, list, K);
    RI_LAUNCHED("ri_gemm_digits");
    return ri_gemm_f32_listed(X, ldx, w32, ldw, C, ldc, M, N, K, list.rows, stream);
}

// The slices of K in which ri_gemm_digits takes a product of M rows that have digits to be made first, 0 where 64-bit sums (ri_gemm_f32) take
// less time.  Both times, us, fitted to 834 measured triples of sizes, rows and slices (12 weights from 1024 x 1024 to 28672 x 4096, 24 to 1,024
// rows, weights from memory, normally distributed; 6 % off, 64-bit sums 13 %): a chunk of 32 values of K takes a block that has its unit to itself 0.89, and
// 0.95 for each of more; the weight's digits come at 4.3 TB/s; the slices' sums are written and read; 18 and 0.0046 for a thousand values of A are the
// split and the two launches behind the product; a unit of the 64-bit kernel takes 0.0023 for 16 x 16 results and a value of K, and 10 beside.  What is so chosen takes
// 1.1 % more on average than the best of each size; furthest from it are 64 rows of 5120 x 3072 (63 us in 64-bit sums, 46 in six slices) and
// 64 of 4096 x 14336 (118 us in six slices, 107 in sixteen).
extern "C" int ri_gemm_digits_plan(int M, int N, int K) {
    if (M < 24 || M > 65535 || (long long)M * N > (1ll << 30) || N < 32 || N % 32 || K < 256 || K % 32 || K > MAX_K) return 0;
    const int chunks = K / 32;
    const long long whole = (long long)((N + 127) / 128 + 7) / 8 * 8 * ((M + 63) / 64);
    int best = 0;
    float least = 0.f;
    for (int parts = 1; parts <= 16 && chunks / parts >= 8; ++parts) {
        const long long blocks = whole * parts;
        if (parts > 1 && (blocks > 2048 || (long long)parts * M * N > (1 << 25))) break;
        const int turns = (chunks + parts - 1) / parts;
        float t = fmaxf((float)turns * (blocks <= 256 ? 0.89f : 0.95f * (float)((blocks + 255) / 256)), (float)N * (float)K * (5.f / 4.3e6f));
        if (parts > 1) t += 5.3f + (float)M * (float)N * (float)(16 * parts + 4) / 8.5e6f;
        if (best == 0 || t < least) { best = parts; least = t; }
    }
    int mt = 0, nt = 0;
    ri_gemm_f32_tile(M, N, &mt, &nt);
    const float units = (float)((((long long)(M + mt - 1) / mt) * ((N + nt - 1) / nt) + 255) / 256) * (float)(mt * nt) / 256.f;
    const float sums64 = fmaxf(units * (float)K * 0.0023f, (float)N * (float)K * (4.f / 4.5e6f)) + 10.f;
    return least + 18.f + (float)M * (float)K * 4.6e-6f < sums64 ? best : 0;
}
