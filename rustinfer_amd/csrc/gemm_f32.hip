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

// Up to eight rows: a tile of the instruction holds eight rows and eight columns of W twice, once for each of two turns of K.
// Lanes r < 8 of A and W hold the values of K of wave w, lanes r >= 8 those of wave w + 4, so the tile's upper left
// quarter is the one wave's sum and the lower right the other's (the other two are not read): four waves do what the eight of
// the kernel above do, in the same order, and a block takes 8 NT columns, so that a product of 2,048 columns gives every
// compute unit a block and no lane loads what another has.  D turns of each wave are under way at a time.  What bounds it is the
// one pass over W.  Measured, us, 6 rows, tiles of 16 rows (half of them no row of the product) with loads that the compiled loop waited for / this
// kernel: 2048 x 2048 10.3 / 6.7, 3072 x 2048 10.8 / 10.2, 16384 x 2048 41 / 31 (134 MB: 4.3 TB/s),
// 2048 x 8192 33 / 17.6, 128256 x 2048 264 / 193 (5.4 TB/s).
// SWIGLU: W is [2N, K] (gate rows, then up rows), a block's two tiles are the gate's and the up rows of the same eight columns, and
// C = silu(gate) * up of the rounded sums, in place of the activation's kernel (six requests generating 12 tokens at the 1B sizes 32.81 -> 32.64 ms:
// two streams of eight rows take most of what the launch of 4.3 us gives back).
template <int NT, int D, bool SWIGLU = false>
__global__ __launch_bounds__(256) void gemm_f32_few_kernel(
        const float* __restrict__ A, int lda, const float* __restrict__ W, int ldw,
        float* __restrict__ C, int ldc, int M, int N, int K) {
    constexpr int TURN = 256;
    __shared__ double sums[8][8][NT * 8];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int r = lane & 7, second = (lane >> 3) & 1, g = lane >> 4;
    static_assert(!SWIGLU || NT == 2, "a tile of gate rows and one of up rows");
    constexpr int COLS = SWIGLU ? 8 : NT * 8;
    const int n0 = (int)blockIdx.x * COLS;
    const char* abase = reinterpret_cast<const char*>(A + wave * 32);
    const char* wbase = reinterpret_cast<const char*>(W + (size_t)n0 * ldw + wave * 32);
    const char* ubase = SWIGLU ? reinterpret_cast<const char*>(W + ((size_t)N + n0) * ldw + wave * 32) : wbase;     // of the last tile
    const int kl = second * 128 + 4 * g;
    const uint32_t arow = ((uint32_t)min(r, M - 1) * (uint32_t)lda + kl) * 4;
    uint32_t wrow[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) wrow[j] = ((uint32_t)min((SWIGLU ? 0 : j * 8) + r, N - 1 - n0) * (uint32_t)ldw + kl) * 4;
    f64x4_t acc[NT] = {};
    auto ask = [&](int turn, float4 (&a)[2], float4 (&w)[2][NT]) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const size_t at = ((size_t)turn * TURN + 16 * u) * 4;
#pragma unroll
            for (int j = 0; j < NT; ++j) w[u][j] = ld_stream16<float4>((j == NT - 1 ? ubase : wbase) + at + wrow[j]);
            a[u] = *reinterpret_cast<const float4*>(abase + at + arow);
        }
    };
    auto add = [&](const float4 (&a)[2], const float4 (&w)[2][NT]) {
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
    // turns that are whole for both halves of the lanes
    const int left = K - wave * 32 - 160;
    const int whole = left >= 0 ? left / TURN + 1 : 0;
    float4 a[D][2], w[D][2][NT];
    if (whole >= D) {
        int turn = 0;
#pragma unroll
        for (int d = 0; d < D; ++d) ask(d, a[d], w[d]);
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
        for (int turn = 0; turn < whole; ++turn) {
            ask(turn, a[0], w[0]);
            add(a[0], w[0]);
        }
    }
    if (wave * 32 + whole * TURN < K) {          // a turn that ends within the lanes' chunks, or before the second half's
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const bool in = wave * 32 + whole * TURN + 16 * u + kl < K;
            const size_t at = ((size_t)whole * TURN + 16 * u) * 4;
#pragma unroll
            for (int j = 0; j < NT; ++j)
                w[0][u][j] = in ? *reinterpret_cast<const float4*>((j == NT - 1 ? ubase : wbase) + at + wrow[j]) : make_float4(0.f, 0.f, 0.f, 0.f);
            a[0][u] = in ? *reinterpret_cast<const float4*>(abase + at + arow) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        add(a[0], w[0]);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 2; ++e) sums[wave + 4 * second][4 * e + g][j * 8 + r] = second ? acc[j][2 + e] : acc[j][e];
    __syncthreads();
    auto sum = [&](int row, int col) {
        double v = sums[0][row][col];
#pragma unroll
        for (int i = 1; i < 8; ++i) v += sums[i][row][col];
        return (float)v;
    };
    for (int e = threadIdx.x; e < 8 * COLS; e += 256) {
        const int row = e / COLS, col = e % COLS;
        float v = sum(row, col);
        if (SWIGLU) v = v / (1.f + expf(-v)) * sum(row, 8 + col);
        if (row < M && n0 + col < N) C[(size_t)row * ldc + n0 + col] = v;
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

// The form of gemm_f32_few_kernel: 0: 8 columns a block and 4 turns under way, 1: 16 and 2, 2: 16 and 1, 3: 24 and 1.  Above 4,096 columns
// the one whose rounds of 256 blocks take the least (*cost: in rounds of 8 columns a block); with fewer columns a block the rows of A
// are read more often.  Measured, us, forms 0 / 2 / 3 at 1 and 8 rows: 6144 x 4096 20.7 26.4 / 26.7 29.7 / 21.9 22.9, 16384 x 2048
// 27.7 35.4 / 27.9 30.7 / 30.6 33.4, 12288 x 4096 37 48 / 40 43 / 37 41, 28672 x 4096 81 108 / 84 93 / 85 92, 128256 x 1024 95 134 / 97
// 113 / 92 107; 0 / 1: 2048 x 8192 16 19 / 24 28, 4096 x 4096 14.8 18.6 / 16.1 17.1, 4096 x 14336 49 64 / 49 56.  (Two forms by
// columns alone, before: 6144 x 4096 29, 16384 x 2048 29 32, 4096 x 14336 49 64.)
static int few_form(int M, int N, int K, float* cost) {
    auto rounds = [&](int columns) { return (float)(((N + columns - 1) / columns + 255) / 256); };
    const float one = rounds(8) * (0.96f + 0.0225f * (float)M + (K < 1024 ? 0.1f : 0.f));
    const float two = rounds(16) * 2.f, three = rounds(24) * 2.8f;
    *cost = fminf(one, fminf(two, three));
    if (N <= 4096) return M > 4 && N > 2048 && K >= 1536 && !(K >= 8192 && (K & (K - 1)) == 0) ? 1 : 0;
    return one == *cost ? 0 : two < three ? 2 : 3;
}

// Whether up to four rows go to the kernel of FMAs, gemm_rows_f32: it reads a kilobyte of a row of W at a time, the tiles 64 bytes
// of each of 16 places, which costs more the longer the rows are.  But where rows begin a power of two apart its long reads meet on the same
// channels of memory, and there it pays only against rounds of blocks that are far from full.  Measured, us, 1 and 4 rows, gemm_rows_f32 / the best form of
// the tiles: 5120 x 3072 16.6 18.6 / 17.4 19.3, 5120 x 5120 23.7 27.1 / 28.5 30.5, 27648 x 5120 97 107 / 120 130, 12288 x 6912 60 68 / 68 71,
// 128256 x 1536 129 141 / 146 155, 2560 x 11008 35 40 / 37 40, 7000 x 4096 25.1 26.6 / 25.9 27.4; not taken: 12288 x 1536 18.4 21.8 / 17.7
// 18.9, 28672 x 4096 95 98 / 81 87, 16384 x 2048 34 37 / 28 29, 4096 x 3072 14.9 16.3 / 12.8 14.4, 2048 x 8192 21 24 / 16 17.
static bool gemm_f32_rows_pay(int M, int N, int K, int ldw) {
    if (M > 4) return false;
    if ((ldw & (ldw - 1)) == 0) {
        float cost = 0.f;
        few_form(M, N, K, &cost);
        return N > 4096 && ((K == 2048 && N > 65536) || (K >= 4096 && cost > 1.1f * (float)N / 2048.f));
    }
    if (N > 4096) return K > 2048 || (K > 1024 && N > 32768) || (K >= 768 && K % 128 != 0);
    return N > 2048 && K >= (N > 3072 ? 7168 : 5120);
}

// The kernel that ri_gemm_f32 takes: -1 gemm_rows_f32, 0 to 3 the form of gemm_f32_few_kernel, 4 the tiles of 16 rows and more.
extern "C" int ri_gemm_f32_form(int M, int N, int K, int ldw) {
    if (gemm_f32_rows_pay(M, N, K, ldw)) return -1;
    // (of 5 to 8 rows with a K that ends inside a turn, wide products stay with the tiles of 16 rows: 12288 x 900 16.9 -> 15.5)
    if (M > 8 || (M > 4 && N > 4096 && K >= 768 && K % 128 != 0)) return 4;
    float cost = 0.f;
    return few_form(M, N, K, &cost);
}

// Whether up to eight rows' gate and up product takes ri_gemm_f32_swiglu rather than ri_gemm_f32 and the activation's kernel: not where gemm_rows_f32
// has that product to itself, but for rows of up to 3,072 values whose rounds of blocks are full.  Measured, us, 1 and 4 rows, two kernels / this:
// 8192 x 3072 46.7 50.3 / 43.8 45.9, 9728 x 2560 40.4 44.2 / 42.4 45.4, 6912 x 2560 29.6 34.6 / 36.1 38.4, 13824 x 5120 98 109 / 128 137, 18944 x 3584
// 92 98 / 107 115, 14336 x 4096 83 90 / 82 85, 8192 x 2048 29.7 30.9 / 29.0 29.8.
extern "C" int ri_gemm_f32_swiglu_pays(int M, int I, int K, int ldw) {
    if (M > 8) return 0;
    const bool full = (float)((I + 2047) / 2048) * 2048.f <= 1.03f * (float)I;
    return !(K > 2048 && gemm_f32_rows_pay(M, 2 * I, K, ldw) && (K > 3072 || !full));
}

// C[M, N] = silu(A . gate^T) * (A . up^T) of up to eight rows, W = [gate; up] of 2N rows: what the tiles of ri_gemm_f32 and the activation's
// kernel give, bit for bit.
extern "C" int ri_gemm_f32_swiglu(const float* A, int lda, const float* W, int ldw, float* C, int ldc,
                                  int M, int N, int K, hipStream_t stream) {
    RI_REQUIRE(M >= 1 && M <= 8 && N > 0 && K > 0 && K % 4 == 0, "ri_gemm_f32_swiglu: needs 1 to 8 rows and K %% 4 == 0 (M=%d N=%d K=%d)", M, N, K);
    RI_REQUIRE(lda >= K && ldw >= K && ldc >= N && lda % 4 == 0 && ldw % 4 == 0 && lda <= (1 << 24) && ldw <= (1 << 24),
               "ri_gemm_f32_swiglu: leading dimensions must be >= K, multiples of 4 and at most 2^24");
    RI_REQUIRE(A && W && C && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0 && N <= (1 << 26), "ri_gemm_f32_swiglu: null or unaligned pointer, or N=%d", N);
    gemm_f32_few_kernel<2, 1, true><<<(N + 7) / 8, 256, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K);
    RI_LAUNCHED("ri_gemm_f32_swiglu");
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
        switch (form) {
            case -1: return ri_gemm_rows_f32(A, lda, W, ldw, C, ldc, M, N, K, stream);
            case 0: gemm_f32_few_kernel<1, 4><<<(N + 7) / 8, 256, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K); break;
            case 1: gemm_f32_few_kernel<2, 2><<<(N + 15) / 16, 256, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K); break;
            case 2: gemm_f32_few_kernel<2, 1><<<(N + 15) / 16, 256, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K); break;
            default: gemm_f32_few_kernel<3, 1><<<(N + 23) / 24, 256, 0, stream>>>(A, lda, W, ldw, C, ldc, M, N, K); break;
        }
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
