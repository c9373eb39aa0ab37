// gemm_f32: C[M, N] = A[M, K] . W[N, K]^T of 32-bit operands with 64-bit sums, on the 64-bit matrix
// instruction v_mfma_f64_16x16x4_f64: a 32-bit value is exact in 64 bits and a product of two as
// well, so the arithmetic is that of a 64-bit FMA loop.  What bounds it is that instruction (64 cycles
// for 2,048 operations: 78.6 TFLOP/s over the chip) or, for few rows, the one pass over W.
//
// The instruction is slow next to what feeds it: a wave that owns 64 x 64 results asks for 8 KiB in
// 4,096 cycles.  So nothing passes through LDS on the way in: every lane reads 16 bytes of K of its row
// of A and of W straight into registers, and the four
// steps of such 16 bytes take the K values {4g + s} of the four lane groups g, for A and W alike.  (A chunk is asked for
// before the one ahead of it is multiplied, but under conditions of the lanes, for which the compiled loop waits for
// every load before it multiplies: what covers a trip to memory is the unit's other waves.)  The
// waves of a block share one tile of results and take 32 values of K in turn, whatever the tile; their 64-bit sums meet in
// LDS once, in the order of the waves, so a row's result does not depend on the other rows or on the tile.  (Products
// of up to four rows, gemm_rows_f32, add in another order: the same to the rounding of a 64-bit sum.)
// Blocks of one column tile run on one XCD (consecutive block ids go around the eight of them), so a
// tile's weights pass through one L2.  K % 4 == 0, rows 16-byte aligned.
//
// Against the FMA kernels with 64-bit sums that were here before, us: 600 rows of 2048 x 8192 1451 -> 366
// (55 TFLOP/s), 256 rows of 16384 x 2048 596 -> 308, 100 rows of 2048 x 2048 296 -> 27, 64 rows of
// 28672 x 4096 801 -> 275, 16 rows of 16384 x 2048 76 -> 41, 8 rows 47 -> 35 (134 MB: 20 at 6.9 TB/s).
#include "common.h"

typedef double f64x4_t __attribute__((ext_vector_type(4)));

// MT x NT tiles of 16 x 16 results a block, WAVES waves that share K, chunks of 16 U values of K (U = 1: two of them, one
// after the other, are a wave's turn of 32).
// STREAM: W is read once (a single row of tiles), past the caches.
template <int MT, int NT, int WAVES, int U, bool STREAM>
__global__ __launch_bounds__(WAVES * 64) void gemm_f32_kernel(
        const float* __restrict__ A, int lda, const float* __restrict__ W, int ldw,
        float* __restrict__ C, int ldc, int M, int N, int K, int mtiles, int ntiles) {
    constexpr int KC = 16 * U, TURN = WAVES * 32, K1 = U == 1 ? KC : TURN, K2 = U == 1 ? TURN : 2 * TURN;
    static_assert(U == 1 || U == 2, "a wave's turn of K is 32 values");
    __shared__ double sums[WAVES][16][NT * 16];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int xcd = (int)blockIdx.x & 7, turn = (int)blockIdx.x >> 3;
    const int nt = (turn / mtiles) * 8 + xcd, mt = turn % mtiles;
    if (nt >= ntiles) return;
    const int m0 = mt * MT * 16, n0 = nt * NT * 16;
    const float* arow[MT];
    const float* wrow[NT];
#pragma unroll
    for (int i = 0; i < MT; ++i) arow[i] = A + (size_t)min(m0 + i * 16 + r, M - 1) * lda + 4 * g;
#pragma unroll
    for (int j = 0; j < NT; ++j) wrow[j] = W + (size_t)min(n0 + j * 16 + r, N - 1) * ldw + 4 * g;
    f64x4_t acc[MT][NT] = {};
    auto ask = [&](int k0, float4 (&a)[U][MT], float4 (&w)[U][NT]) {
        const bool whole = k0 + KC <= K;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + 16 * u;
            const bool in = whole || k + 4 * g < K;
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                w[u][j] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (in) w[u][j] = STREAM ? ld_stream16<float4>(wrow[j] + k) : *reinterpret_cast<const float4*>(wrow[j] + k);
            }
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                a[u][i] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (in) a[u][i] = *reinterpret_cast<const float4*>(arow[i] + k);
            }
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
    float4 a0[U][MT], w0[U][NT], a1[U][MT], w1[U][NT];
    int k = wave * 32;
    if (k < K) ask(k, a0, w0);
    for (; k < K; k += K2) {
        const int k1 = k + K1, k2 = k + K2;
        if (k1 < K) ask(k1, a1, w1);
        add(a0, w0);
        if (k1 < K) {
            if (k2 < K) ask(k2, a0, w0);
            add(a1, w1);
        }
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
            if (m < M && n < N) C[(size_t)m * ldc + n] = (float)v;
        }
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

// The rows and columns of the tile that ri_gemm_f32 takes for M rows and N columns.
extern "C" void ri_gemm_f32_tile(int M, int N, int* rows, int* columns) {
    const F32Tile& t = F32_TILES[f32_tile(M, N)];
    *rows = 16 * t.mt;
    *columns = 16 * t.nt;
}

// The 32-bit product of any number of rows (K % 4 == 0, operands and rows 16-byte aligned).
extern "C" int ri_gemm_f32(const float* A, int lda, const float* W, int ldw, float* C, int ldc,
                           int M, int N, int K, hipStream_t stream) {
    RI_REQUIRE(M >= 1 && N > 0 && K > 0 && K % 4 == 0, "ri_gemm_f32: needs rows and K %% 4 == 0 (M=%d N=%d K=%d)", M, N, K);
    RI_REQUIRE(lda >= K && ldw >= K && ldc >= N && lda % 4 == 0 && ldw % 4 == 0, "ri_gemm_f32: leading dimensions must be >= K and multiples of 4");
    RI_REQUIRE(A && W && C && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0, "ri_gemm_f32: null or unaligned pointer");
    RI_REQUIRE(N <= (1 << 26), "ri_gemm_f32: N=%d exceeds the grid limit", N);
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
