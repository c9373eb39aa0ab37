// gemm_digits: C[M, N] = A[M, K] . W[N, K]^T of 32-bit operands in exact integer sums, on the 8-bit matrix instruction, for
// the 32-bit path's prompts.  Each row of A and of W is brought to whole numbers of 40 bits: x = q 2^(e - 39), e the least exponent
// that holds the row's largest magnitude, and q to five digits of eight bits, base 256, from -128 to 127.  A product of two rows
// is then 25 products of digits; the 15 whose weight is at least 256^4 are summed, each in 32-bit integers that cannot
// overflow (K <= 26,000), and put together in 64-bit integers, which the rounding to 32-bit floats ends.
// So a result has one rounding, as a 64-bit sum has (gemm_f32.hip): a row's values are cut at 2^-40 of its largest and the ten
// products left out lie below 2^-38 of the two rows' largest, where a 32-bit result's own rounding is 2^-25 of itself.  Integer sums
// have no order: a row's bits depend neither on the tile, nor on the slices of K, nor on the other rows.  Against 64 bits,
// 600 rows of 16384 x 2048, normally distributed: 2.5306e-8 in the 2-norm, as 64-bit sums have; beyond half a unit of a result's last place
// by 1.1e-11 of the largest result at most.
//
// Rows whose values spread too far for that (more of them below 2^-13 of the largest than above, zeros aside) and rows that hold an
// infinity or a NaN are taken by 64-bit FMAs instead, from the 32-bit values themselves; a weight with such a row gets no
// digits at all.
//
// Digits lie as the matrix instruction takes them: [rows / 32][K / 32][5][64 lanes][16 bytes], lane 32 h + r holding k = 16 h .. 16 h + 15 of
// row r.  A block of eight waves makes 64 x 128 results: a stage of 32 values of K (30 KiB) goes straight into LDS while
// the stage before is multiplied; two such blocks fit a unit.  What bounds it: the instruction at the clock that the card's power leaves it (a
// loop of it alone reaches 4.7 POP/s on zeros and 3.4 on random digits; this kernel 2.9 and 2.3).  Measured, us, 64-bit sums / this without
// the split of A: 600 rows of 16384 x 2048 663 / 264, 3072 x 2048 143 / 53, 2048 x 2048 96 / 46, 2048 x 8192 354 / 141; 194 rows
// 252 / 102 (16384 x 2048), 135 / 58 (2048 x 8192); 89 rows 111 / 55, 86 / 35.  Tiles of 128 x 128 and 64 x 64, of four and eight waves, and
// three stages: 0 to 10 % slower.  Six digits and 21 products: 341 for the first.
#include "common.h"
#include <float.h>
#include <limits.h>

typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x16_t __attribute__((ext_vector_type(16)));

namespace {

constexpr int DIGITS = 5, PIECE = DIGITS * 1024;              // bytes of 32 rows by 32 values of K
constexpr int NOT_SPLIT = INT_MIN;                            // in the place of a row's exponent
constexpr int MAX_K = 26000;                                  // 5 products of at most 2^14 a value of K in 32-bit sums

// s_waitcnt: at most n loads under way, whatever is asked of LDS
constexpr int loads_imm(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }

// Rows of values: those of X (gate == 0), or silu(X[:, k]) * X[:, gate + k], the exponential in 32 bits and the rest in 64, not
// rounded to 32 in between (beyond their range it is infinite all the same).
struct Rows {
    const float* x;
    int ld, gate;
    __device__ __forceinline__ void at(int row, int k, double (&v)[4]) const {
        const float* p = x + (size_t)row * ld + k;
        const float4 f = *reinterpret_cast<const float4*>(p);
        v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
        if (gate) {
            const float4 g = *reinterpret_cast<const float4*>(p + gate);
            const float u[4] = {g.x, g.y, g.z, g.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[i] = v[i] * (double)u[i] / (1.0 + (double)expf(-(float)v[i]));
                if (!(fabs(v[i]) <= (double)FLT_MAX)) v[i] = (double)(float)v[i];
            }
        }
    }
};

__device__ __forceinline__ float to_float(long long sum, int ea, int ew) {
    return (float)((double)sum * __longlong_as_double((long long)(1023 + ea + ew - 46) << 52));
}

// A row without digits, by one wave: a 64-bit sum, the lanes' shares in the order of K.
__device__ __forceinline__ float row_dot(const Rows& a, int m, const float* __restrict__ w, int K) {
    const int lane = threadIdx.x & 63;
    double v = 0.0;
    for (int k = lane * 4; k < K; k += 256) {
        double x[4];
        a.at(m, k, x);
        const float4 y = *reinterpret_cast<const float4*>(w + k);
        v = fma(x[0], (double)y.x, v);
        v = fma(x[1], (double)y.y, v);
        v = fma(x[2], (double)y.z, v);
        v = fma(x[3], (double)y.w, v);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return (float)v;
}

// The digits and exponents of rows.  A block a row (rows of a last tile beyond the end are zeros), sixteen values a thread and turn,
// read for the largest, then for the digits, the first turn's kept.  Four rows that follow each other run on one XCD, so that the 16 bytes a row
// leaves of each line meet in one L2.  Bound by waiting: 600 rows of 2,048 6.6 us, of 8,192 with the activation 28 (36 with every turn computed twice).
template <bool GATE>
__global__ __launch_bounds__(512) void digits_split_kernel(Rows a, int rows, int K, uint8_t* __restrict__ planes, int* __restrict__ exps) {
    __shared__ uint32_t largest[8];
    __shared__ int above[8];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, waves = blockDim.x >> 6;
    const int b = blockIdx.x, row = (b >> 5) * 32 + (b & 7) * 4 + ((b >> 3) & 3);
    const bool in = row < rows;
    if (!GATE) a.gate = 0;
    auto high = [](double v) { return (uint32_t)(__double_as_longlong(v) >> 32) & 0x7fffffffu; };      // exponent and 20 bits
    uint32_t most = 0;
    const int first = threadIdx.x * 16;
    double kept[4][4] = {};                                      // of the first turn, the only one up to 8,192 values
    auto look = [&](const double (&v)[4]) { most = max(most, max(max(high(v[0]), high(v[1])), max(high(v[2]), high(v[3])))); };
    if (in && first < K)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            a.at(row, first + 4 * q, kept[q]);
            look(kept[q]);
        }
    if (in)
        for (int k = first + blockDim.x * 16; k < K; k += blockDim.x * 16)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                double v[4];
                a.at(row, k + 4 * q, v);
                look(v);
            }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) most = max(most, (uint32_t)__shfl_xor((int)most, o, 64));
    if (lane == 0) largest[wave] = most;
    __syncthreads();
    for (int i = 0; i < waves; ++i) most = max(most, largest[i]);
    const bool finite = most < 0x7ff00000u;
    int e = 0;
    if (most && finite) {
        // the largest, its cut-off bits and a 128th more are below 2^e: its first digit, with what the others' signs carry into it, is at most 127
        const uint32_t up = most + (((most & 0xfffffu) | 0x100000u) >> 7) + 2;
        e = (int)(up >> 20) - 1022;
    }
    const double scale = __longlong_as_double((long long)(1023 + 39 - e) << 52);
    uint8_t* out = planes + (size_t)(row >> 5) * (K / 32) * PIECE + (row & 31) * 16;
    const uint32_t small = most >= (13u << 20) ? most - (13u << 20) : 0u;
    int balance = 0;
    for (int k = first; k < K; k += blockDim.x * 16) {
        uint32_t d[DIGITS][4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            double v[4] = {0.0, 0.0, 0.0, 0.0};
            if (in && finite) {
                if (k == first)
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[j] = kept[q][j];
                else a.at(row, k + 4 * q, v);
            }
            uint32_t lo[4], hi[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                balance += high(v[j]) >= small ? 1 : high(v[j]) ? -1 : 0;
                const long long n = (long long)rint(v[j] * scale) + 0x80808080ll;
                lo[j] = (uint32_t)n ^ 0x80808080u;               // four digits, signed bytes
                hi[j] = (uint32_t)(n >> 32);                     // the first
            }
            // bytes of four values to four values a digit: digits 0 and 1, 2 and 3 of two values each, then of four
            const uint32_t p01 = __builtin_amdgcn_perm(lo[1], lo[0], 0x05010400u), q01 = __builtin_amdgcn_perm(lo[1], lo[0], 0x07030602u);
            const uint32_t p23 = __builtin_amdgcn_perm(lo[3], lo[2], 0x05010400u), q23 = __builtin_amdgcn_perm(lo[3], lo[2], 0x07030602u);
            d[0][q] = __builtin_amdgcn_perm(p23, p01, 0x05040100u);
            d[1][q] = __builtin_amdgcn_perm(p23, p01, 0x07060302u);
            d[2][q] = __builtin_amdgcn_perm(q23, q01, 0x05040100u);
            d[3][q] = __builtin_amdgcn_perm(q23, q01, 0x07060302u);
            d[4][q] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(hi[3], hi[2], 0x00000400u), __builtin_amdgcn_perm(hi[1], hi[0], 0x00000400u), 0x05040100u);
        }
        uint8_t* o = out + (size_t)(k >> 5) * PIECE + ((k >> 4) & 1) * 512;
#pragma unroll
        for (int i = 0; i < DIGITS; ++i) *reinterpret_cast<uint4*>(o + i * 1024) = make_uint4(d[i][0], d[i][1], d[i][2], d[i][3]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) balance += __shfl_xor(balance, o, 64);
    if (lane == 0) above[wave] = balance;
    __syncthreads();
    if (threadIdx.x == 0) {
        int sum = 0;
        for (int i = 0; i < waves; ++i) sum += above[i];
        exps[row] = !in ? 0 : finite && sum >= 0 ? e : NOT_SPLIT;
    }
}

// 2 x 4 waves of 32 x 32 results.  blockIdx.y: the slice of K, `part` chunks of 32 values; with several, sums
// [parts][M][N] are left in P for digits_sum_kernel, else the results in C.
__global__ __launch_bounds__(512, 4) void gemm_digits_kernel(
        const uint8_t* __restrict__ A, const int* __restrict__ ea, Rows rows, const uint8_t* __restrict__ W, const int* __restrict__ ew,
        const float* __restrict__ w32, int ldw, float* __restrict__ C, int ldc, long long* __restrict__ P,
        int M, int N, int K, int part, int mblocks, int nblocks) {
    constexpr int WM = 2, WN = 4, WAVES = WM * WN, FRAGS = (WM + WN) * DIGITS, PER = (FRAGS + WAVES - 1) / WAVES, STAGE = FRAGS * 1024;
    __shared__ __align__(16) uint8_t lds[2 * STAGE];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave % WM, wn = wave / WM;
    // the row blocks of one block of columns run on one XCD (consecutive block ids go around the eight of them)
    const int id = (int)blockIdx.x, turn = id >> 3;
    const int nb = (turn / mblocks) * 8 + (id & 7), mb = turn % mblocks;
    if (nb >= nblocks) return;
    const int mtiles = (M + 31) / 32, ntiles = N / 32, chunks = K / 32;
    // a wave brings in four of the stage's 30 kilobytes, the last two of them twice; tiles beyond the end are read (clamped), never stored
    const uint8_t* from[PER];
    int to[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int f = min(wave * PER + i, FRAGS - 1), t = f / DIGITS;
        const int tile = t < WM ? min(mb * WM + t, mtiles - 1) : min(nb * WN + t - WM, ntiles - 1);
        from[i] = (t < WM ? A : W) + (size_t)tile * chunks * PIECE + f % DIGITS * 1024 + lane * 16;
        to[i] = f * 1024;
    }
    auto fetch = [&](int c, int at) {
#pragma unroll
        for (int i = 0; i < PER; ++i)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(from[i] + (size_t)c * PIECE),
                (__attribute__((address_space(3))) void*)(lds + at + to[i]), 16, 0, 0);
    };
    // acc[s]: the products of digits i and j with i + j = 4 + s
    i32x16_t acc[DIGITS] = {};
    const int c0 = blockIdx.y * part, c1 = min(chunks, c0 + part);
    if (c0 < c1) fetch(c0, 0);
    int at = 0;
    for (int c = c0; c < c1; ++c) {
        __builtin_amdgcn_s_waitcnt(loads_imm(0));                // this wave's part of the stage has arrived, and behind the barrier everyone's;
        __builtin_amdgcn_s_barrier();                            // all have read the other one
        asm volatile("" ::: "memory");
        if (c + 1 < c1) fetch(c + 1, STAGE - at);
        const i32x4_t* la = reinterpret_cast<const i32x4_t*>(lds + at + wm * PIECE) + lane;
        const i32x4_t* lw = reinterpret_cast<const i32x4_t*>(lds + at + (WM + wn) * PIECE) + lane;
        i32x4_t b[DIGITS];
#pragma unroll
        for (int j = DIGITS - 1; j >= 0; --j) b[j] = lw[j * 64];
#pragma unroll
        for (int i = 0; i < DIGITS; ++i) {
            const i32x4_t a = la[i * 64];
#pragma unroll
            for (int j = DIGITS - 1 - i; j < DIGITS; ++j)
                acc[i + j - (DIGITS - 1)] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b[j], acc[i + j - (DIGITS - 1)], 0, 0, 0);
        }
        at = STAGE - at;
    }
    // result (row 8 (i / 4) + 4 (lane / 32) + i % 4, column lane % 32) of a tile lies in element i
    const int n = (nb * WN + wn) * 32 + (lane & 31), m0 = (mb * WM + wm) * 32;
    if ((nb * WN + wn) * 32 >= N || m0 >= M) return;
    const int fw = ew[n];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int m = m0 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
        if (m >= M) continue;
        long long v = acc[DIGITS - 1][i];
#pragma unroll
        for (int s = DIGITS - 2; s >= 0; --s) v = v * 256 + acc[s][i];
        if (P) P[((size_t)blockIdx.y * M + m) * N + n] = v;
        else if (ea[m] != NOT_SPLIT) C[(size_t)m * ldc + n] = to_float(v, ea[m], fw);
    }
    if (P) return;
    uint32_t left = (uint32_t)__ballot(m0 + (lane & 31) < M && ea[min(m0 + (lane & 31), M - 1)] == NOT_SPLIT);     // a bit a row, the same in all lanes
    for (; left; left &= left - 1) {
        const int m = m0 + __builtin_ctz(left), first = (nb * WN + wn) * 32;
        for (int j = 0; j < 32; ++j) {
            const float v = row_dot(rows, m, w32 + (size_t)(first + j) * ldw, K);
            if (lane == 0) C[(size_t)m * ldc + first + j] = v;
        }
    }
}

// The slices' sums, added up and rounded once: a block 256 columns of a row.
__global__ __launch_bounds__(256) void digits_sum_kernel(const long long* __restrict__ P, int parts, const int* __restrict__ ea, Rows rows,
                                                         const int* __restrict__ ew, const float* __restrict__ w32, int ldw,
                                                         float* __restrict__ C, int ldc, int M, int N, int K) {
    const int m = blockIdx.y, n = blockIdx.x * 256 + threadIdx.x, e = ea[m];
    if (e == NOT_SPLIT) {
        const int first = blockIdx.x * 256 + (threadIdx.x >> 6) * 64;
        for (int j = first; j < min(first + 64, N); ++j) {
            const float v = row_dot(rows, m, w32 + (size_t)j * ldw, K);
            if ((threadIdx.x & 63) == 0) C[(size_t)m * ldc + j] = v;
        }
        return;
    }
    if (n >= N) return;
    long long v = 0;
    for (int p = 0; p < parts; ++p) v += P[((size_t)p * M + m) * N + n];
    C[(size_t)m * ldc + n] = to_float(v, e, ew[n]);
}

}  // namespace

// Bytes of the digits of `rows` rows of K values (whole tiles of 32 rows), and how many exponents go with them.
extern "C" long long ri_digits_bytes(int rows, int K) { return (long long)((rows + 31) / 32) * (K / 32) * PIECE; }

extern "C" int ri_digits_max_k() { return MAX_K; }

// Digits and exponents (one a row of whole tiles of 32; INT_MIN: a row that has none) of X[rows, K], or with gate > 0 of
// silu(X[:, :K]) * X[:, gate : gate + K].
extern "C" int ri_digits_split(const float* X, int ld, int rows, int K, int gate, void* planes, int* exps, hipStream_t stream) {
    RI_REQUIRE(rows >= 1 && K >= 32 && K % 32 == 0 && K <= MAX_K, "ri_digits_split: needs K %% 32 == 0 and at most %d (rows=%d K=%d)", MAX_K, rows, K);
    RI_REQUIRE(ld >= K + gate && ld % 4 == 0 && gate >= 0 && gate % 4 == 0 && (gate == 0 || gate >= K), "ri_digits_split: bad leading dimension or columns");
    RI_REQUIRE(X && planes && exps && (uintptr_t)X % 16 == 0 && (uintptr_t)planes % 16 == 0, "ri_digits_split: null or unaligned pointer");
    RI_REQUIRE(rows <= (1 << 22), "ri_digits_split: rows=%d exceed the grid limit", rows);
    const int threads = min(512, (K / 16 + 63) / 64 * 64), blocks = (rows + 31) / 32 * 32;
    const Rows a{X, ld, gate};
    if (gate) digits_split_kernel<true><<<blocks, threads, 0, stream>>>(a, rows, K, (uint8_t*)planes, exps);
    else digits_split_kernel<false><<<blocks, threads, 0, stream>>>(a, rows, K, (uint8_t*)planes, exps);
    RI_LAUNCHED("ri_digits_split");
    return 0;
}

// C[M, N] from the digits of A (of the rows X, ldx, gate: see ri_digits_split) and of W (w32: its 32-bit values).  parts > 1: slices of K, sums [parts][M][N].
extern "C" int ri_gemm_digits(const void* A, const int* ea, const float* X, int ldx, int gate, const void* W, const int* ew,
                              const float* w32, int ldw, float* C, int ldc, long long* sums, int parts,
                              int M, int N, int K, hipStream_t stream) {
    RI_REQUIRE(M >= 1 && N >= 32 && N % 32 == 0 && K >= 32 && K % 32 == 0 && K <= MAX_K,
               "ri_gemm_digits: needs N and K in multiples of 32, K at most %d (M=%d N=%d K=%d)", MAX_K, M, N, K);
    RI_REQUIRE(A && ea && X && W && ew && w32 && C && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0 && (uintptr_t)X % 16 == 0
               && (uintptr_t)w32 % 16 == 0, "ri_gemm_digits: null or unaligned pointer");
    RI_REQUIRE(ldx >= K + gate && ldx % 4 == 0 && gate >= 0 && gate % 4 == 0 && ldw >= K && ldw % 4 == 0 && ldc >= N, "ri_gemm_digits: bad leading dimensions");
    RI_REQUIRE(parts >= 1 && parts <= 64 && (parts == 1 || sums), "ri_gemm_digits: parts=%d", parts);
    const int mblocks = (M + 63) / 64, nblocks = (N + 127) / 128, chunks = K / 32;
    const long long blocks = (long long)((nblocks + 7) / 8 * 8) * mblocks;
    RI_REQUIRE(blocks * parts < (1 << 22) && M <= 65535, "ri_gemm_digits: M=%d N=%d exceed the grid limit", M, N);
    const Rows a{X, ldx, gate};
    gemm_digits_kernel<<<dim3((unsigned)blocks, parts), 512, 0, stream>>>((const uint8_t*)A, ea, a, (const uint8_t*)W, ew, w32, ldw, C, ldc,
        parts > 1 ? sums : nullptr, M, N, K, (chunks + parts - 1) / parts, mblocks, nblocks);
    RI_LAUNCHED("ri_gemm_digits");
    if (parts > 1) {
        digits_sum_kernel<<<dim3((N + 255) / 256, M), 256, 0, stream>>>(sums, parts, ea, a, ew, w32, ldw, C, ldc, M, N, K);
        RI_LAUNCHED("ri_gemm_digits");
    }
    return 0;
}

extern "C" void ri_gemm_f32_tile(int M, int N, int* rows, int* columns);      // gemm_f32.hip

// The slices of K in which ri_gemm_digits takes a product of M rows that have digits to be made first, 0 where 64-bit sums (ri_gemm_f32) take
// less time.  Both times, us, fitted to 1,050 measured triples of sizes, rows and slices (12 weights from 768 x 3072 to 28672 x 4096, 12 to 1,024
// rows, weights from memory; 8 % off): a chunk of 32 values of K takes a block that has its unit to itself 0.82, and
// 0.77 for each of more; the weight's digits come at 5.5 TB/s; the slices' sums are written and read; a unit of the 64-bit kernel takes
// 0.0021 for 16 x 16 results and a value of K.  The slices so found cost 0.8 % on average against the best of each
// size, and near the line (24 to 64 rows, narrow weights) products that would gain up to 13 % stay where they were.
extern "C" int ri_gemm_digits_plan(int M, int N, int K) {
    if (M < 24 || M > 65535 || N < 32 || N % 32 || K < 256 || K % 32 || K > MAX_K) return 0;
    const int chunks = K / 32;
    const long long whole = (long long)((N + 127) / 128 + 7) / 8 * 8 * ((M + 63) / 64);
    int best = 0;
    float least = 0.f;
    for (int parts = 1; parts <= 16 && chunks / parts >= 8; ++parts) {
        const long long blocks = whole * parts;
        if (parts > 1 && (blocks > 2048 || (long long)parts * M * N > (1 << 25))) break;
        const int turns = (chunks + parts - 1) / parts;
        float t = fmaxf((float)turns * (blocks <= 256 ? 0.82f : 0.77f * (float)((blocks + 255) / 256)), (float)N * (float)K * (5.f / 5.5e6f));
        if (parts > 1) t += 4.1f + (float)M * (float)N * (float)(16 * parts + 4) / 5.0e6f;
        if (best == 0 || t < least) { best = parts; least = t; }
    }
    int mt = 0, nt = 0;
    ri_gemm_f32_tile(M, N, &mt, &nt);
    const float units = (float)((((long long)(M + mt - 1) / mt) * ((N + nt - 1) / nt) + 255) / 256) * (float)(mt * nt) / 256.f;
    const float sums64 = fmaxf(units * (float)K * 0.0021f, (float)N * (float)K * (4.f / 5.0e6f));
    return least + 3.1f + 4.f < sums64 + 4.f ? best : 0;
}
