// gemm_f32: C[M, N] = A[M, K] . W[N, K]^T of 32-bit operands with 64-bit sums, on the 64-bit matrix
// instruction v_mfma_f64_16x16x4_f64: a 32-bit value is exact in 64 bits and a product of two as
// well, so the arithmetic is that of a 64-bit FMA loop.  What bounds it is that instruction (64 cycles
// for 2,048 operations: 78.6 TFLOP/s over the chip) or, for few rows, the one pass over W.
//
// The instruction is slow next to what feeds it: a wave that owns 64 x 64 results asks for 8 KiB in
// 4,096 cycles.  So nothing passes through LDS on the way in: every lane reads 16 bytes of K of its row
// of A and of W straight into registers, and the four
// steps of such 16 bytes take the K values {4g + s} of the four lane groups g, for A and W alike.  A chunk is asked for
// two ahead of the one that is multiplied; nothing on that way depends on the lane, so the compiled loop waits for a
// chunk's own loads only.  The
// waves of a block share one tile of results and take 32 values of K in turn, whatever the tile; their 64-bit sums meet in
// LDS once, in the order of the waves, so a row's result does not depend on the other rows or on the tile.  (Up to four rows of
// products that gemm_f32_rows_pay names go to gemm_rows_f32, gemm.hip, which adds in another order: the same to the rounding of a 64-bit sum.)
// Blocks of one column tile run on one XCD (consecutive block ids go around the eight of them), so a
// tile's weights pass through one L2.  K % 4 == 0, rows 16-byte aligned.
//
// (Prompts of 24 rows or more go to gemm_digits.hip where the weight's digits are laid out.)  What is left to bound the large products: other instructions hold the 64-bit matrix instruction up (a loop of it alone reaches 72
// TFLOP/s on random operands, one with the widening of one operand value an instruction, as in tiles of 32 x 32, 61),
// and that is what they take.  Loads waited for under conditions of the lanes before, now, us: 600 rows of 16384 x 2048 707, 662
// (61 TFLOP/s), of 2048 x 8192 364, 333, of 2048 x 2048 100, 93; 230 rows 268, 250 / 154, 137 / 44, 39; 37 rows of
// 16384 x 2048 67, 60; 13 rows 43, 37.  (As FMA kernels with 64-bit sums: 600 rows of 2048 x 8192 1451.)
#include "common.h"
#include <algorithm>
#include <type_traits>

extern "C" int ri_gemm_tiled(const void* A, int lda, const void* W, int ldw, void* C, int ldc,
                             int M, int N, int K, int in_dtype, int out_dtype, hipStream_t stream);      // gemm.hip
extern "C" int ri_gemm_rows_f32(const float* A, int lda, const float* W, int ldw, float* C, int ldc,
                                int M, int N, int K, hipStream_t stream);                               // gemm.hip

typedef double f64x4_t __attribute__((ext_vector_type(4)));

// MT x NT tiles of 16 x 16 results a block, WAVES waves that share K, chunks of 16 U values of K (U = 1: two of them, one
// after the other, are a wave's turn of 32).
// STREAM: W is read once (a single row of tiles), past the caches.
// The tile with number `id`.  LISTED: of the rows of A and C only the M whose numbers stand in list[1] and on.
template <int MT, int NT, int WAVES, int U, bool STREAM, bool LISTED>
__device__ __forceinline__ void f32_tile_of(
        const float* __restrict__ A, int lda, const float* __restrict__ W, int ldw,
        float* __restrict__ C, int ldc, int M, int N, int K, int mtiles, int ntiles, const int* __restrict__ list, int id) {
    constexpr int KC = 16 * U, TURN = WAVES * 32;
    static_assert(U == 1 || U == 2, "a wave's turn of K is 32 values");
    __shared__ double sums[WAVES][16][NT * 16];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int xcd = id & 7, turn = id >> 3;
    const int nt = (turn / mtiles) * 8 + xcd, mt = turn % mtiles;
    if (nt >= ntiles) return;
    const int m0 = mt * MT * 16, n0 = nt * NT * 16;
    // the block's first rows, the same in all lanes, and each lane's rows as 32-bit distances in bytes from there (listed rows, which may lie
    // anywhere, as 64-bit ones from the first of all)
    const char* abase = reinterpret_cast<const char*>(LISTED ? A : A + (size_t)m0 * lda);
    const char* wbase = reinterpret_cast<const char*>(W + (size_t)n0 * ldw);
    typename std::conditional<LISTED, size_t, uint32_t>::type arow[MT];
    uint32_t wrow[NT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int row = min(i * 16 + r, M - 1 - m0);
        if constexpr (LISTED) arow[i] = ((size_t)list[1 + m0 + row] * lda + 4 * g) * 4;
        else arow[i] = ((uint32_t)row * (uint32_t)lda + 4 * g) * 4;
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) wrow[j] = ((uint32_t)min(j * 16 + r, N - 1 - n0) * (uint32_t)ldw + 4 * g) * 4;
    auto of_a = [&](int i, int k) { return *reinterpret_cast<const float4*>(abase + (size_t)k * 4 + arow[i]); };
    auto of_w = [&](int j, int k) {
        const char* p = wbase + (size_t)k * 4 + wrow[j];
        return STREAM ? ld_stream16<float4>(p) : *reinterpret_cast<const float4*>(p);
    };
    f64x4_t acc[MT][NT] = {};
    auto at = [&](int step) { return wave * 32 + (U == 2 ? step * TURN : (step >> 1) * TURN + (step & 1) * KC); };
    // a whole chunk: no condition of the lanes, so that the loads stay in flight while the chunk ahead is multiplied
    auto ask = [&](int step, float4 (&a)[U][MT], float4 (&w)[U][NT]) {
        const int k0 = at(step);
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int j = 0; j < NT; ++j) w[u][j] = of_w(j, k0 + 16 * u);
#pragma unroll
            for (int i = 0; i < MT; ++i) a[u][i] = of_a(i, k0 + 16 * u);
        }
    };
    auto ask_part = [&](int step, float4 (&a)[U][MT], float4 (&w)[U][NT]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = at(step) + 16 * u;
            const bool in = k + 4 * g < K;
#pragma unroll
            for (int j = 0; j < NT; ++j) w[u][j] = in ? of_w(j, k) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int i = 0; i < MT; ++i) a[u][i] = in ? of_a(i, k) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    auto add = [&](const float4 (&a)[U][MT], const float4 (&w)[U][NT]) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                double x[MT], y[NT];
#pragma unroll
                for (int i = 0; i < MT; ++i) x[i] = (double)(s == 0 ? a[u][i].x : s == 1 ? a[u][i].y : s == 2 ? a[u][i].z : a[u][i].w);
#pragma unroll
                for (int j = 0; j < NT; ++j) y[j] = (double)(s == 0 ? w[u][j].x : s == 1 ? w[u][j].y : s == 2 ? w[u][j].z : w[u][j].w);
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i], y[j], acc[i][j], 0, 0, 0);
            }
    };
    // whole chunks of this wave: step s is whole if at(s) + KC <= K
    int whole = 0;
    const int left = K - wave * 32;
    if (U == 2) whole = left >= 32 ? (left - 32) / TURN + 1 : 0;
    else whole = left < 16 ? 0 : left / TURN * 2 + (left % TURN >= 32 ? 2 : left % TURN >= 16 ? 1 : 0);
    float4 a0[U][MT], w0[U][NT], a1[U][MT], w1[U][NT];
    // One way into the loop, both chunks asked for: at a place that can be reached with fewer loads under way, the compiled
    // code would wait for more of them.  The scheduler's barriers keep the second chunk's conversions, and so the wait for it,
    // behind the first's products.
    if (whole >= 2) {
        int step = 0;
        ask(0, a0, w0);
        ask(1, a1, w1);
        for (; step + 4 <= whole; step += 2) {
            add(a0, w0);
            ask(step + 2, a0, w0);
            __builtin_amdgcn_sched_barrier(0);
            add(a1, w1);
            ask(step + 3, a1, w1);
            __builtin_amdgcn_sched_barrier(0);
        }
        add(a0, w0);                             // two or three are left
        if (step + 2 < whole) ask(step + 2, a0, w0);
        __builtin_amdgcn_sched_barrier(0);
        add(a1, w1);
        __builtin_amdgcn_sched_barrier(0);
        if (step + 2 < whole) add(a0, w0);
    } else if (whole == 1) {
        ask(0, a0, w0);
        add(a0, w0);
    }
    if (at(whole) < K) {                         // and perhaps a part of one
        ask_part(whole, a0, w0);
        add(a0, w0);
    }
    // result (row 4 i + g, column r) of a tile lies in element i of lane 16 g + r
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        if (i) __syncthreads();
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) sums[wave][4 * e + g][j * 16 + r] = acc[i][j][e];
        __syncthreads();
        for (int e = threadIdx.x; e < 16 * NT * 16; e += WAVES * 64) {
            const int row = e / (NT * 16), col = e % (NT * 16);
            double v = sums[0][row][col];
#pragma unroll
            for (int w = 1; w < WAVES; ++w) v += sums[w][row][col];
            const int m = m0 + i * 16 + row, n = n0 + col;
            if (m < M && n < N) C[(size_t)(LISTED ? list[1 + m] : m) * ldc + n] = (float)v;
        }
    }
}

// A tile a block.  LISTED: the rows' number, list[0], is not known to the launch: as many blocks as the chip
// holds take the tiles in turn (an empty list 4.6 us, where a block for each tile of 600 rows of 16384 columns took 5.6).
template <int MT, int NT, int WAVES, int U, bool STREAM, bool LISTED = false>
__global__ __launch_bounds__(WAVES * 64, 4) void gemm_f32_kernel(
        const float* __restrict__ A, int lda, const float* __restrict__ W, int ldw,
        float* __restrict__ C, int ldc, int M, int N, int K, int mtiles, int ntiles, const int* __restrict__ list = nullptr) {
    if constexpr (LISTED) {
        M = list[0];
        mtiles = (M + MT * 16 - 1) / (MT * 16);
        for (int id = (int)blockIdx.x; id < (ntiles + 7) / 8 * 8 * mtiles; id += (int)gridDim.x) {
            f32_tile_of<MT, NT, WAVES, U, STREAM, true>(A, lda, W, ldw, C, ldc, M, N, K, mtiles, ntiles, list, id);
            __syncthreads();                     // the sums in LDS have been read
        }
    } else {
        f32_tile_of<MT, NT, WAVES, U, STREAM, false>(A, lda, W, ldw, C, ldc, M, N, K, mtiles, ntiles, nullptr, (int)blockIdx.x);
    }
}

// Up to eight rows: a tile of the instruction holds eight rows and eight columns of W twice, once for each of two shares of K.
// The eight waves of the kernel above are halves of four here: lanes r < 8 of A and W hold the values of K of its wave 2 w,
// lanes r >= 8 those of 2 w + 1, so the tile's upper left quarter is the one's sum and the lower right the other's (the other two are not
// read), made in the same order, and a block takes 8 NT columns, so that a product of 2,048 columns gives every
// compute unit a block and no lane loads what another has.  D turns of each wave are under way at a time.  What bounds it is the
// one pass over W.  A load takes 128 bytes of each of eight rows, a whole line: the lanes' second half asks for what the first half multiplies
// behind its own 64 bytes, and the two change places on the way to the instruction (with 64 bytes of 16 places a load every line was
// asked for twice).  Measured, us, 1 and 8 rows, 64 bytes / this:
// 2048 x 2048 7.3 7.6 / 6.9 7.1, 16384 x 2048 28.9 30.5 / 28.1 27.6, 2048 x 8192 16.3 18.9 / 16.9 18.1, 12288 x 1536 17.9 19.6 / 16.5 18.0, 8 rows
// of 4096 x 14336 55.8 / 45.5 (235 MB: 5.2 TB/s), 13824 x 2560 43.4 / 35.7, 27648 x 5120 140 / 114, 128256 x 2048 203 / 186 (5.7 TB/s).
// SWIGLU: W is [2N, K] (gate rows, then up rows), a block's two tiles are the gate's and the up rows of the same eight columns, and
// C = silu(gate) * up of the rounded sums, in place of the activation's kernel (8 rows of 2 x 8192 x 2048 33.2 / 30.3, 2 x 14336 x 4096 93 / 84).
//
// A norm between two such products has no kernel of its own, as in gemm.hip.  RESID (the product before it): C is the residual stream, C += sums, and what is left for the
// product behind it are rows C * weight of the norm, 32-bit, and the sums of C^2 over the block's columns.  With `scale.ssq` a product finishes such a norm:
// row m of its sums is multiplied by 1 / sqrt(mean of the row's squares + eps), in 64 bits, before it is rounded.  A result then passes two roundings of 32 bits
// where the norm's kernel makes three.
// ROPE: the product is q/k/v: a block's two tiles are eight features of a head's first half and the eight that they turn with; q goes to C, k and v to the pages.
// Each saves a launch of 4.6 to 5.6 us.
enum FewKind { FEW_PLAIN, FEW_SWIGLU, FEW_RESID, FEW_ROPE };
struct FewScale { const float* ssq; int parts; float eps; };                            // ssq [M, parts]
struct FewResid { const float* w; float* a; float* ssq; };                              // w [N]; a [M, N]; ssq [M, blocks]
struct FewRope {
    const float* cos_t; const float* sin_t;        // [positions][hd / 2]
    const int* positions; const int* row_of_token; // of a row of A
    const int* table; int max_blocks;              // block table [rows][max_blocks]
    float* kc; float* vc;                          // k [pages][Hkv][page][hd], v [pages][Hkv][hd][page]
    int H, Hkv, hd, page;
};
template <int NT, int D, FewKind KIND = FEW_PLAIN>
__global__ __launch_bounds__(256) void gemm_f32_few_kernel(
        const float* __restrict__ A, int lda, const float* __restrict__ W, int ldw,
        float* __restrict__ C, int ldc, int M, int N, int K, const FewScale scale, const FewResid resid, const FewRope rope) {
    constexpr int TURN = 256;
    constexpr bool TWO = KIND == FEW_SWIGLU || KIND == FEW_ROPE;       // two streams of eight rows of W
    __shared__ double sums[8][8][NT * 8];
    __shared__ double factors[8];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int r = lane & 7, second = (lane >> 3) & 1, g = lane >> 4;
    static_assert(!TWO || NT == 2, "a tile of each");
    static_assert(KIND != FEW_RESID || NT <= 2, "a row's columns of a block lie in 8 or 16 lanes");
    constexpr int COLS = TWO ? 8 : NT * 8;
    // the block's first row of W, and rows from there to the other stream's
    const int per_head = KIND == FEW_ROPE ? rope.hd >> 4 : 1;
    const int head = KIND == FEW_ROPE ? (int)blockIdx.x / per_head : 0, feature = KIND == FEW_ROPE ? ((int)blockIdx.x - head * per_head) * 8 : 0;
    const int n0 = KIND == FEW_ROPE ? head * rope.hd + feature : (int)blockIdx.x * COLS;
    const size_t apart = KIND == FEW_ROPE ? (size_t)(rope.hd >> 1) : (size_t)N;
    const char* abase = reinterpret_cast<const char*>(A + wave * 64);
    const char* wbase = reinterpret_cast<const char*>(W + (size_t)n0 * ldw + wave * 64);
    const char* ubase = TWO ? reinterpret_cast<const char*>(W + (apart + n0) * ldw + wave * 64) : wbase;     // of the last tile
    // of a wave's 64 values of a turn: the 16-byte pieces of W that a lane asks for lie at wl and wl + 32, the ones of A that it multiplies at al and al + 16
    const int wl = second * 16 + 4 * g, al = second * 32 + 4 * g;
    const uint32_t arow = ((uint32_t)min(r, M - 1) * (uint32_t)lda + al) * 4;
    uint32_t wrow[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) wrow[j] = ((uint32_t)min((TWO ? 0 : j * 8) + r, N - 1 - n0) * (uint32_t)ldw + wl) * 4;
    // What the end needs beside the sums is asked for behind the first turns of W.  This thread's result is row `row`, column `col` of the block's.
    const int row = (int)threadIdx.x / COLS, col = (int)threadIdx.x % COLS;
    const bool mine = row < M && n0 + col < N;       // (an own bound of `row`: M <= 8)
    const bool scaled = KIND != FEW_RESID && scale.ssq != nullptr;
    float4 squares[2] = {};                          // of rows `wave` and `wave + 4`
    float x_own = 0.f, w_own = 0.f, cs = 1.f, sn = 0.f;
    int pos = 0, entry = -1, blk = -1;
    auto early = [&]() {
        if (scaled) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
                if (wave + 4 * i < M && lane * 4 < scale.parts) squares[i] = *reinterpret_cast<const float4*>(scale.ssq + (size_t)(wave + 4 * i) * scale.parts + lane * 4);
        }
        if constexpr (KIND == FEW_RESID) {
            if (mine) {
                x_own = C[(size_t)row * ldc + n0 + col];
                w_own = resid.w[n0 + col];
            }
        }
        if constexpr (KIND == FEW_ROPE) {
            if (wave == 0) {                         // (64 results: the first wave's)
                // scalar loads, which do not stand behind the weights
#pragma unroll
                for (int m = 0; m < 8; ++m) {
                    if (m >= M) break;
                    const int b = rope.row_of_token[m], p = rope.positions[m];
                    const int at = b >= 0 ? rope.table[(size_t)b * rope.max_blocks + p / rope.page] : -1;
                    if (row == m) { entry = b; pos = p; blk = at; }
                }
                if (entry >= 0) {
                    cs = rope.cos_t[(size_t)pos * (rope.hd >> 1) + feature + col];
                    sn = rope.sin_t[(size_t)pos * (rope.hd >> 1) + feature + col];
                }
            }
        }
    };
    f64x4_t acc[NT] = {};
    auto ask = [&](int turn, float4 (&a)[2], float4 (&w)[2][NT]) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const size_t at = (size_t)turn * TURN * 4;
#pragma unroll
            for (int j = 0; j < NT; ++j) w[u][j] = ld_stream16<float4>((j == NT - 1 ? ubase : wbase) + at + 128 * u + wrow[j]);
            a[u] = *reinterpret_cast<const float4*>(abase + at + 64 * u + arow);
        }
    };
    // the lanes' first half has the pieces of its own two steps in w[0] of both halves, the second in w[1] of both
    auto swapped = [&](float& p, float& q) {
        const int sent = __float_as_int(second ? p : q), got = __builtin_amdgcn_mov_dpp(sent, 0x128, 0xf, 0xf, true);       // lane ^ 8
        if (second) p = __int_as_float(got);
        else q = __int_as_float(got);
    };
    auto add = [&](const float4 (&a)[2], float4 (&w)[2][NT]) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            swapped(w[0][j].x, w[1][j].x);
            swapped(w[0][j].y, w[1][j].y);
            swapped(w[0][j].z, w[1][j].z);
            swapped(w[0][j].w, w[1][j].w);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const double x = (double)(s == 0 ? a[u].x : s == 1 ? a[u].y : s == 2 ? a[u].z : a[u].w);
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const double y = (double)(s == 0 ? w[u][j].x : s == 1 ? w[u][j].y : s == 2 ? w[u][j].z : w[u][j].w);
                    acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x, y, acc[j], 0, 0, 0);
                }
            }
    };
    // turns of which the wave's 64 values are all there
    const int left = K - wave * 64 - 64;
    const int whole = left >= 0 ? left / TURN + 1 : 0;
    float4 a[D][2], w[D][2][NT];
    if (whole >= D) {
        int turn = 0;
#pragma unroll
        for (int d = 0; d < D; ++d) ask(d, a[d], w[d]);
        early();
        for (; turn + 2 * D <= whole; turn += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                add(a[d], w[d]);
                ask(turn + d + D, a[d], w[d]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        const int more = whole - turn - D;       // of the next D turns, so many are there
#pragma unroll
        for (int d = 0; d < D; ++d) {
            add(a[d], w[d]);
            if (d < more) ask(turn + d + D, a[d], w[d]);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (d < more) add(a[d], w[d]);
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
        early();
        for (int turn = 0; turn < whole; ++turn) {
            ask(turn, a[0], w[0]);
            add(a[0], w[0]);
        }
    }
    if (const int k0 = wave * 64 + whole * TURN; k0 < K) {           // a turn that ends within the wave's values
        const size_t at = (size_t)whole * TURN * 4;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const bool in_w = k0 + 32 * u + wl < K, in_a = k0 + 16 * u + al < K;
#pragma unroll
            for (int j = 0; j < NT; ++j)
                w[0][u][j] = in_w ? *reinterpret_cast<const float4*>((j == NT - 1 ? ubase : wbase) + at + 128 * u + wrow[j]) : make_float4(0.f, 0.f, 0.f, 0.f);
            a[0][u] = in_a ? *reinterpret_cast<const float4*>(abase + at + 64 * u + arow) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        add(a[0], w[0]);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 2; ++e) sums[2 * wave + second][4 * e + g][j * 8 + r] = second ? acc[j][2 + e] : acc[j][e];
    if (scaled) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int m = wave + 4 * i;
            if (m >= M) break;
            double s = ((double)squares[i].x + (double)squares[i].y) + ((double)squares[i].z + (double)squares[i].w);
            for (int p = 256 + lane * 4; p < scale.parts; p += 256) {
                const float4 v = *reinterpret_cast<const float4*>(scale.ssq + (size_t)m * scale.parts + p);
                s += ((double)v.x + (double)v.y) + ((double)v.z + (double)v.w);
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
            if (lane == 0) factors[m] = 1.0 / sqrt(s / K + (double)scale.eps);
        }
    }
    __syncthreads();
    auto sum = [&](int m, int c) {
        double v = sums[0][m][c];
#pragma unroll
        for (int i = 1; i < 8; ++i) v += sums[i][m][c];
        return (float)(scaled ? v * factors[m] : v);
    };
    if (threadIdx.x >= 8 * COLS) return;             // COLS <= 32
    if constexpr (KIND == FEW_RESID) {
        float v = 0.f;
        if (mine) {
            v = x_own + sum(row, col);
            C[(size_t)row * ldc + n0 + col] = v;
            resid.a[(size_t)row * N + n0 + col] = v * w_own;
        }
        float sq = v * v;
#pragma unroll
        for (int o = COLS / 2; o > 0; o >>= 1) sq += __shfl_xor(sq, o, 64);
        if (row < M && col == 0) resid.ssq[(size_t)row * gridDim.x + blockIdx.x] = sq;
    } else if constexpr (KIND == FEW_ROPE) {
        if (row >= M || entry < 0) return;           // a padding token
        const float p = sum(row, col), q = sum(row, 8 + col);
        const float first = p * cs - q * sn, behind = p * sn + q * cs;
        const int half = rope.hd >> 1, i = feature + col, slot = pos % rope.page;
        if (head < rope.H) {
            float* to = C + (size_t)row * ldc + n0 + col;
            to[0] = first;
            to[half] = behind;
        } else if (blk >= 0) {
            const int group = (head - rope.H) % rope.Hkv;
            const size_t at = ((size_t)blk * rope.Hkv + group) * rope.page * rope.hd;
            if (head < rope.H + rope.Hkv) {
                float* to = rope.kc + at + (size_t)slot * rope.hd + i;
                to[0] = first;
                to[half] = behind;
            } else {
                float* to = rope.vc + at + (size_t)i * rope.page + slot;
                to[0] = p;
                to[(size_t)half * rope.page] = q;
            }
        }
    } else if (mine) {
        float v = sum(row, col);
        if (KIND == FEW_SWIGLU) v = v / (1.f + expf(-v)) * sum(row, 8 + col);
        C[(size_t)row * ldc + n0 + col] = v;
    }
}

// The tile of a product: the fewest results that a compute unit gets, ceil(blocks / 256) tiles of MT x NT
// (a unit's matrix instructions are what its blocks share, however many of them it holds), with the small
// tiles counted a little dearer for the operands that they ask for more often.  Measured, us, tiles of
// 16x16 / 32x16 / 16x32 / 32x32 / 48x32: 24 rows of 2048 x 2048 11.5 / 16.5 / 18.0 / - / -; 24 rows of
// 4096 x 14336 145 / 93 / 120 / - / -; 100 rows of 3072 x 2048 - / - / 40.7 / 45.5 / -; 160 rows of
// 2048 x 8192 - / - / 140 / 154 / -; 33 rows of 16384 x 2048 - / - / 77 / 84 / 63; 256 rows of
// 16384 x 2048 - / - / 360 / 308 / - (64x64: 328).
struct F32Tile { int mt, nt; float dear; };
static const F32Tile F32_TILES[] = {{2, 2, 1.f}, {3, 2, 1.f}, {2, 1, 1.1f}, {1, 2, 1.12f}, {1, 1, 1.25f}};

static int f32_tile(int M, int N) {
    int best = 0;
    float least = 0.f;
    for (int i = 0; i < (int)(sizeof(F32_TILES) / sizeof(F32_TILES[0])); ++i) {
        const F32Tile& t = F32_TILES[i];
        const long long blocks = (long long)((M + 16 * t.mt - 1) / (16 * t.mt)) * ((N + 16 * t.nt - 1) / (16 * t.nt));
        const float cost = (float)((blocks + 255) / 256) * t.mt * t.nt * t.dear;
        if (i == 0 || cost < least) { best = i; least = cost; }
    }
    return best;
}

// A launch holds fewer than 2^32 threads, 8 M blocks of 512: larger products take several, of whole rows of tiles each.
template <int MT, int NT, int U>
static void launch_f32(const float* A, int lda, const float* W, int ldw, float* C, int ldc, int M, int N, int K, hipStream_t stream) {
    const int ntiles = (N + 16 * NT - 1) / (16 * NT), across = (ntiles + 7) / 8 * 8;
    const int most = ((1 << 23) - 1) / across * 16 * MT;
    for (int m0 = 0; m0 < M; m0 += most) {
        const int m = min(M - m0, most), mtiles = (m + 16 * MT - 1) / (16 * MT);
        const float* a = A + (size_t)m0 * lda;
        float* c = C + (size_t)m0 * ldc;
        if (mtiles == 1) gemm_f32_kernel<MT, NT, 8, U, true><<<across, 512, 0, stream>>>(a, lda, W, ldw, c, ldc, m, N, K, mtiles, ntiles);
        else gemm_f32_kernel<MT, NT, 8, U, false><<<across * mtiles, 512, 0, stream>>>(a, lda, W, ldw, c, ldc, m, N, K, mtiles, ntiles);
    }
}

// The rows of A[M, K] and C[M, N] whose numbers stand in list[1] and on, list[0] of them (on the device, 0 to M): what ri_gemm_f32 gives for them, in the tiles that it
// takes for M rows.
extern "C" int ri_gemm_f32_listed(const float* A, int lda, const float* W, int ldw, float* C, int ldc, int M, int N, int K,
                                  const int* list, hipStream_t stream) {
    RI_REQUIRE(M >= 1 && N > 0 && K > 0 && K % 4 == 0 && lda >= K && ldw >= K && ldc >= N && lda % 4 == 0 && ldw % 4 == 0 && ldw <= (1 << 24),
               "ri_gemm_f32_listed: needs rows, K %% 4 == 0 and leading dimensions >= K and multiples of 4 (M=%d N=%d K=%d)", M, N, K);
    RI_REQUIRE(A && W && C && list && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0, "ri_gemm_f32_listed: null or unaligned pointer");
    RI_REQUIRE((long long)M * ((N + 15) / 16 + 7) < (1ll << 31), "ri_gemm_f32_listed: M=%d N=%d exceed the grid limit", M, N);
    const F32Tile& t = F32_TILES[f32_tile(M, N)];
    const int mtiles = (M + 16 * t.mt - 1) / (16 * t.mt), ntiles = (N + 16 * t.nt - 1) / (16 * t.nt), blocks = std::min((ntiles + 7) / 8 * 8 * mtiles, 512);
    switch (f32_tile(M, N)) {
        case 0: gemm_f32_kernel<2, 2, 8, 2, false, true><<<blocks, 512, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K, mtiles, ntiles, list); break;
        case 1: gemm_f32_kernel<3, 2, 8, 1, false, true><<<blocks, 512, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K, mtiles, ntiles, list); break;
        case 2: gemm_f32_kernel<2, 1, 8, 2, false, true><<<blocks, 512, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K, mtiles, ntiles, list); break;
        case 3: gemm_f32_kernel<1, 2, 8, 2, false, true><<<blocks, 512, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K, mtiles, ntiles, list); break;
        default: gemm_f32_kernel<1, 1, 8, 2, false, true><<<blocks, 512, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K, mtiles, ntiles, list); break;
    }
    RI_LAUNCHED("ri_gemm_f32_listed");
    return 0;
}

// The rows and columns of the tile that ri_gemm_f32 takes for M rows and N columns (of gemm_f32_kernel: up to eight rows, the tiles
// of gemm_f32_few_kernel hold eight, and gemm_rows_f32 has none; see ri_gemm_f32_form).
extern "C" void ri_gemm_f32_tile(int M, int N, int* rows, int* columns) {
    const F32Tile& t = F32_TILES[f32_tile(M, N)];
    *rows = 16 * t.mt;
    *columns = 16 * t.nt;
}

// The form of gemm_f32_few_kernel: 0: 8 columns a block and 4 turns under way, 1 (up to 4,096 columns) and 2 (above): 16 and 2, 3: 24 and 2.  Above 4,096 columns
// the one whose rounds of 256 blocks take the least (*cost: in rounds of 8 columns a block); with fewer columns a block the rows of A
// are read more often.  Measured, us, 8 / 16 / 24 columns at 1 and 8 rows: 6144 x 4096 19.8 24.5 / 26.8 28.1 / 21.0 21.5, 16384 x 2048
// 27.0 32.2 / 27.8 28.4 / 30.2 30.6, 12288 x 4096 35 46 / 43 45 / 38 39, 28672 x 4096 78 102 / 89 95 / 84 88, 128256 x 1024 89 122 / 100 111 / 88 94.
// Up to there 8 and 16 at 8 rows: 4096 x 4096 17.4 / 18.6, 4096 x 8192 32.5 / 33.2 (these two take the slower), 4096 x 14336 54 / 49, 4096 x 16384 63 / 55,
// 3072 x 8192 31.6 / 28.2, 2560 x 8192 31.4 / 27.4, 3072 x 3584 at 0.89 of the time with 16; 2048 x 8192 18.6 / 27.3: one round of half the blocks.
static float few_rounds(int N, int columns) { return (float)(((N + columns - 1) / columns + 255) / 256); }
static float few_cost8(int M, int N, int K) { return few_rounds(N, 8) * (0.96f + 0.0225f * (float)M + (K < 1024 ? 0.1f : 0.f)); }
static int few_form(int M, int N, int K, float* cost) {
    const float one = few_cost8(M, N, K);
    const float two = few_rounds(N, 16) * 2.f, three = few_rounds(N, 24) * 2.8f;
    *cost = fminf(one, fminf(two, three));
    if (N <= 4096) return M > 4 && N > 2048 && K >= 1536 && !(N < 2560 && K >= 8192 && (K & (K - 1)) == 0) ? 1 : 0;
    return one == *cost ? 0 : two < three ? 2 : 3;
}

// Whether up to four rows go to the kernel of FMAs, gemm_rows_f32: it reads a kilobyte of a row of W at a time, the tiles 128 bytes
// of each of eight rows.  Measured, time of gemm_rows_f32 / of the tiles' form, at 1, 2, 3 and 4 rows, for 23 numbers of columns and 11 lengths of rows:
// whole tiles (N % 8 == 0) and chunks (K % 128 == 0), rows no power of two apart:
//     up to 4,096 columns 1.06 to 1.29 everywhere; 8,192 < N <= 20,480 1.00 to 1.50 (10240 x 5120 1.20 1.21 1.20 1.21)
//     5,120 to 8,192 columns, K > 3072: 0.88 to 1.05 at one row (7168 x 6912 0.88, 5120 x 9216 0.90, 8192 x 5120 1.05), 0.94 to 1.08 at two (from 4,608 values on
//     0.94 to 1.05), 0.95 to 1.10 at three, 1.01 to 1.13 at four; shorter rows 0.97 to 1.35
//     24,576 columns and more: K <= 2304 0.95 to 1.46; longer ones 0.87 to 1.15 (65536 x 4608 0.92 0.87 0.94 0.94, 36864 x 6912 0.95 0.97 0.97 0.98,
//     28672 x 3072 1.15 0.99 1.07 1.05, 50304 x 5120 0.99 0.97 0.90 0.91)
// Where rows begin a power of two apart its long reads meet on the same channels of memory, and there it pays only against rounds of blocks that are far from
// full: us, 1 and 4 rows, gemm_rows_f32 / tiles, taken: 5120 x 4096 at 4 rows 21.4 / 20.3, 9216 x 8192 72 / 64, 128256 x 2048 173 179 / 164 173; not
// 28672 x 4096 96 102 / 78 85, 16384 x 2048 34 37 / 27 27, 12288 x 4096 39 43 / 38 38, 2048 x 8192 21 24 / 17 17.
// Sizes with remainders keep the line that was drawn for rows of 64 bytes a load (5001 x 2304, 2049 x 5124, 4111 x 772 are on its side).
static bool gemm_f32_long_rows(int M, int N, int K, int ldw) {
    if (M > 4) return false;
    if ((ldw & (ldw - 1)) == 0) {
        float cost = 0.f;
        few_form(M, N, K, &cost);
        return N > 4096 && ((K == 2048 && N > 65536) || (K >= 4096 && cost > 1.1f * (float)N / 2048.f));
    }
    if (N > 4096) return K > 2048 || (K > 1024 && N > 32768) || (K >= 768 && K % 128 != 0);
    return N > 2048 && K >= (N > 3072 ? 7168 : 5120);
}
static bool gemm_f32_rows_pay(int M, int N, int K, int ldw) {
    if (M > 4 || (ldw & (ldw - 1)) == 0 || N % 8 != 0 || K % 128 != 0) return gemm_f32_long_rows(M, N, K, ldw);
    return N > 20480 ? K > 2304 : N > 4096 && N <= 8192 && ((M == 1 && K > 3072) || (M == 2 && K > 4096));
}

// The kernel that ri_gemm_f32 takes: -1 gemm_rows_f32, 0 to 3 the form of gemm_f32_few_kernel, 4 the tiles of 16 rows and more.
extern "C" int ri_gemm_f32_form(int M, int N, int K, int ldw) {
    if (gemm_f32_rows_pay(M, N, K, ldw)) return -1;
    // (of 5 to 8 rows with a K that ends inside a turn, wide products stay with the tiles of 16 rows: 12288 x 900 16.9 -> 15.5)
    if (M > 8 || (M > 4 && N > 4096 && K >= 768 && K % 128 != 0)) return 4;
    float cost = 0.f;
    return few_form(M, N, K, &cost);
}

// Whether up to eight rows' gate and up product takes ri_gemm_f32_swiglu rather than ri_gemm_f32 and the activation's kernel.  Its blocks hold eight columns of each,
// so its rounds of 256 blocks are of 2,048 columns; where rows are long the line is at rounds 8/9 full.  Measured, us, 1 and 4 rows, two kernels / this:
// 9216 x 2304 38.7 42.3 / 33.9 35.0, 9728 x 2560 40 44 / 37 38, 13824 x 2560 55 60 / 49 50, 8192 x 3072 46 51 / 37 38, 14336 x 3584 73 78 / 66 69, 18944 x 3584 93 97 / 91 94,
// 13824 x 5120 100 108 / 97 102, 17408 x 5120 119 127 / 118 125; not taken 6912 x 2560 29.9 35.0 / 31.7 32.4, 2560 x 3588 21.3 23.2 / 24.3 25.7, 6912 x 5120 53 60 / 57 59, 7168 x 3584
// 38.7 43.8 / 39.7 41.5; rows of more than 5,120 values keep the two, 24576 x 6144 183 188 / 182 195 (6144 x 6144 57 63 / 51 53).  Rows a power of two apart: 14336 x 4096 78 87 / 75 77,
// 8192 x 2048 29.6 29.6 / 30.3 30.7.  (Behind a deferred norm the product is always this one.)
extern "C" int ri_gemm_f32_swiglu_pays(int M, int I, int K, int ldw) {
    if (M > 8) return 0;
    const bool full = (I + 2047) / 2048 * 2048 * 8 <= I * 9;
    return !(K > 2048 && gemm_f32_long_rows(M, 2 * I, K, ldw) && (K > 5120 || !full));
}

static bool few_scale_ok(const float* ssq, int parts, float eps) {
    return !ssq || (parts >= 4 && parts % 4 == 0 && eps >= 0.f && (uintptr_t)ssq % 16 == 0);
}

static void launch_few(int form, const float* A, int lda, const float* W, int ldw, float* C, int ldc, int M, int N, int K, const FewScale& scale,
                       hipStream_t stream) {
    if (form == 0) gemm_f32_few_kernel<1, 4><<<(N + 7) / 8, 256, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K, scale, FewResid{}, FewRope{});
    else if (form == 3) gemm_f32_few_kernel<3, 2><<<(N + 23) / 24, 256, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K, scale, FewResid{}, FewRope{});
    else gemm_f32_few_kernel<2, 2><<<(N + 15) / 16, 256, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K, scale, FewResid{}, FewRope{});
}

#define FEW_REQUIRE(who) \
    RI_REQUIRE(M >= 1 && M <= 8 && N > 0 && K > 0 && K % 4 == 0, who ": needs 1 to 8 rows and K %% 4 == 0 (M=%d N=%d K=%d)", M, N, K); \
    RI_REQUIRE(lda >= K && ldw >= K && lda % 4 == 0 && ldw % 4 == 0 && lda <= (1 << 24) && ldw <= (1 << 24), \
               who ": leading dimensions must be >= K, multiples of 4 and at most 2^24"); \
    RI_REQUIRE(A && W && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0 && N <= (1 << 26), who ": null or unaligned pointer, or N=%d", N)

// C[M, N] = silu(A . gate^T) * (A . up^T) of up to eight rows, W = [gate; up] of 2N rows: what the tiles of ri_gemm_f32 and the activation's
// kernel give, bit for bit.  ssq [M, parts] (or null): see ri_gemm_f32_scaled.
extern "C" int ri_gemm_f32_swiglu(const float* A, int lda, const float* W, int ldw, float* C, int ldc,
                                  int M, int N, int K, const float* ssq, int parts, float eps, hipStream_t stream) {
    FEW_REQUIRE("ri_gemm_f32_swiglu");
    RI_REQUIRE(C && ldc >= N && few_scale_ok(ssq, parts, eps), "ri_gemm_f32_swiglu: bad result or partial sums of squares");
    gemm_f32_few_kernel<2, 2, FEW_SWIGLU><<<(N + 7) / 8, 256, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K, FewScale{ssq, parts, eps}, FewResid{}, FewRope{});
    RI_LAUNCHED("ri_gemm_f32_swiglu");
    return 0;
}

// C[M, N] = (A . W^T) of up to eight rows, row m times 1 / sqrt(sum(ssq[m]) / K + eps): ssq [M, parts], a multiple of 4 of them, as ri_gemm_f32_residual leaves them.
extern "C" int ri_gemm_f32_scaled(const float* A, int lda, const float* W, int ldw, float* C, int ldc,
                                  int M, int N, int K, const float* ssq, int parts, float eps, hipStream_t stream) {
    FEW_REQUIRE("ri_gemm_f32_scaled");
    RI_REQUIRE(C && ldc >= N && ssq && few_scale_ok(ssq, parts, eps), "ri_gemm_f32_scaled: bad result or partial sums of squares");
    float cost = 0.f;
    launch_few(few_form(M, N, K, &cost), A, lda, W, ldw, C, ldc, M, N, K, FewScale{ssq, parts, eps}, stream);
    RI_LAUNCHED("ri_gemm_f32_scaled");
    return 0;
}

// Partial sums of squares that ri_gemm_f32_residual leaves of a row of N values: one for 8 or 16 columns a block, whichever of the two takes the
// fewer rounds (24 columns are not among them: their sums lie in no 8 or 16 lanes).  us with the gate/up product behind it, 16 columns for every size that takes 24 elsewhere / this, 1 and
// 4 rows: 5120 x 13824 and 2 x 3840 104 105 / 88 97, 5120 x 5120 and 2 x 13824 129 133 / 121 129, 6144 x 6144 and 2 x 6144 88 91 / 81 87.
extern "C" int ri_gemm_f32_residual_parts(int M, int N, int K) {
    float cost = 0.f;
    const bool eight = N <= 4096 ? few_form(M, N, K, &cost) == 0 : few_cost8(M, N, K) <= few_rounds(N, 16) * 2.f;
    return N / (eight ? 8 : 16);
}

// x[M, N] += A . W^T of up to eight rows, and for the norm behind it (weights norm_w [N]) a[M, N] = x * norm_w and partial sums of x^2, ssq [M, parts].  N % 64 == 0.
extern "C" int ri_gemm_f32_residual(const float* A, int lda, const float* W, int ldw, int M, int N, int K, float* x, const float* norm_w, float* a, float* ssq,
                                    hipStream_t stream) {
    FEW_REQUIRE("ri_gemm_f32_residual");
    RI_REQUIRE(N % 64 == 0 && x && norm_w && a && ssq, "ri_gemm_f32_residual: null pointer, or N=%d", N);
    const FewResid resid{norm_w, a, ssq};
    if (ri_gemm_f32_residual_parts(M, N, K) == N / 8) gemm_f32_few_kernel<1, 4, FEW_RESID><<<N / 8, 256, 0, stream>>>(A, lda, W, ldw, x, N, M, N, K, FewScale{}, resid, FewRope{});
    else gemm_f32_few_kernel<2, 2, FEW_RESID><<<N / 16, 256, 0, stream>>>(A, lda, W, ldw, x, N, M, N, K, FewScale{}, resid, FewRope{});
    RI_LAUNCHED("ri_gemm_f32_residual");
    return 0;
}

// q/k/v [M, (H + 2 Hkv) hd] of up to eight tokens, q and k turned by the token's position over the whole head: q to the first H hd columns of C, k and v to the
// token's page.  Tokens of no request (row_of_token < 0) leave nothing.  ssq: see ri_gemm_f32_scaled, or null.
extern "C" int ri_gemm_f32_qkv_rope(const float* A, int lda, const float* W, int ldw, float* C, int ldc, int M, int K, int H, int Hkv, int hd,
                                    const float* cos_t, const float* sin_t, const int* positions, const int* row_of_token, float* kc, float* vc,
                                    const int* table, int max_blocks, int page, const float* ssq, int parts, float eps, hipStream_t stream) {
    RI_REQUIRE(H >= 1 && Hkv >= 1 && hd >= 16 && hd % 16 == 0 && H <= (1 << 12) && Hkv <= (1 << 12) && hd <= (1 << 12) && page >= 1 && max_blocks >= 1,
               "ri_gemm_f32_qkv_rope: bad sizes H=%d Hkv=%d hd=%d page=%d", H, Hkv, hd, page);
    const int N = (H + 2 * Hkv) * hd;
    FEW_REQUIRE("ri_gemm_f32_qkv_rope");
    RI_REQUIRE(C && ldc >= H * hd && cos_t && sin_t && positions && row_of_token && kc && vc && table && few_scale_ok(ssq, parts, eps),
               "ri_gemm_f32_qkv_rope: null pointer, or bad result or partial sums of squares");
    const FewRope rope{cos_t, sin_t, positions, row_of_token, table, max_blocks, kc, vc, H, Hkv, hd, page};
    gemm_f32_few_kernel<2, 2, FEW_ROPE><<<N / 16, 256, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K, FewScale{ssq, parts, eps}, FewResid{}, rope);
    RI_LAUNCHED("ri_gemm_f32_qkv_rope");
    return 0;
}

// The 32-bit product of any number of rows (K % 4 == 0, operands and rows 16-byte aligned).
extern "C" int ri_gemm_f32(const float* A, int lda, const float* W, int ldw, float* C, int ldc,
                           int M, int N, int K, hipStream_t stream) {
    RI_REQUIRE(M >= 1 && N > 0 && K > 0 && K % 4 == 0, "ri_gemm_f32: needs rows and K %% 4 == 0 (M=%d N=%d K=%d)", M, N, K);
    RI_REQUIRE(lda >= K && ldw >= K && ldc >= N && lda % 4 == 0 && ldw % 4 == 0, "ri_gemm_f32: leading dimensions must be >= K and multiples of 4");
    RI_REQUIRE(A && W && C && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0, "ri_gemm_f32: null or unaligned pointer");
    RI_REQUIRE(N <= (1 << 26), "ri_gemm_f32: N=%d exceeds the grid limit", N);
    // lanes find their rows by 32-bit distances in bytes from the first of up to 48
    if (M <= 4 && (lda > (1 << 24) || ldw > (1 << 24))) return ri_gemm_rows_f32(A, lda, W, ldw, C, ldc, M, N, K, stream);
    if (lda > (1 << 24) || ldw > (1 << 24)) return ri_gemm_tiled(A, lda, W, ldw, C, ldc, M, N, K, RI_F32, RI_F32, stream);
    if (const int form = ri_gemm_f32_form(M, N, K, ldw); form < 4) {
        if (form < 0) return ri_gemm_rows_f32(A, lda, W, ldw, C, ldc, M, N, K, stream);
        launch_few(form, A, lda, W, ldw, C, ldc, M, N, K, FewScale{}, stream);
        RI_LAUNCHED("ri_gemm_f32");
        return 0;
    }
    switch (f32_tile(M, N)) {
        case 0: launch_f32<2, 2, 2>(A, lda, W, ldw, C, ldc, M, N, K, stream); break;
        case 1: launch_f32<3, 2, 1>(A, lda, W, ldw, C, ldc, M, N, K, stream); break;
        case 2: launch_f32<2, 1, 2>(A, lda, W, ldw, C, ldc, M, N, K, stream); break;
        case 3: launch_f32<1, 2, 2>(A, lda, W, ldw, C, ldc, M, N, K, stream); break;
        default: launch_f32<1, 1, 2>(A, lda, W, ldw, C, ldc, M, N, K, stream); break;
    }
    RI_LAUNCHED("ri_gemm_f32");
    return 0;
}
