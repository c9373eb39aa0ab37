// gemm_mid: C[M, N] = A[M, K] . W[N, K]^T for portions of some tens to hundreds of bfloat16 rows against weights
// in tile order ([N/16][K/32][64 lanes][8], see gemm.hip): the steps that hold a prompt's portion beside decoding
// requests, and short prompts.
//
// With that many rows a product of a few thousand columns makes too few tiles of 128 x 128 for 256 compute units,
// so K is divided between blocks (blockIdx.y), each leaving 32-bit partial sums in its own slice of C; the norm or
// the rotation that follows adds them up as it reads them.  SWIGLU: the tiles of a block are as many of the gate
// half and of the up half of a stacked [2N, K] matrix, and C = silu(gate) * up in bfloat16.
//
// A block brings stretches of 64 values of K of its rows and of its weight tiles into a ring of ST stages of LDS
// with loads that write LDS directly, and reads them in the order the matrix instructions take them.  What bounds
// it is LDS (a wave of 32 x 64 results reads 6 KiB for 8 matrix instructions of 16 cycles); measured for
// 28672 x 4096 and 128 rows: 50 us, 45 with all weights from one tile, 38 without the matrix instructions.  A
// deeper ring for the weights alone, another first stretch for each block and loads past the caches gave nothing.
// Measured (us, the GEMM library's kernel / this, alone, without what adds the slices up): 4096 x 14336, 96, 128, 256, 512
// rows 63 75 61 92 / 28 28 39 64; 4096 x 4096 20 22 22 29 / 12 13 16 24; 6144 x 4096 22 25 40 37 / 16 18 25 38; 2048 x 8192
// 19 20 27 34 / 12 13 17 25.  With what follows, and gate/up with SwiGLU: ri_gemm_mid_plan, ops._slices_pay, ops.qkv_split_pays.
#include "common.h"
#include <mutex>

typedef __bf16 mbf16x8_t __attribute__((ext_vector_type(8)));
typedef float mf32x4_t __attribute__((ext_vector_type(4)));

namespace {

constexpr int KS = 2;                         // k-steps of 32 in a stretch: 128 bytes of a row

// s_waitcnt: at most n loads under way, and nothing asked of LDS
constexpr int wait_imm(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4); }

// WM x WN waves of MW x NTW tiles of 16 x 16 results each.
template <int WM, int WN, int MW, int NTW, int ST, bool SWIGLU, typename TO>
__global__ __launch_bounds__(WM * WN * 64) void gemm_mid_kernel(
        const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W,
        TO* __restrict__ C, int ldc, int M, int N, int K, int mblocks, int nblocks, int stretches_per_part,
        size_t part_stride) {
    constexpr int WAVES = WM * WN, BM = WM * MW * 16, BT = WN * NTW;     // rows and weight tiles of a block
    constexpr int XA = BM * KS * 4, XW = BT * KS * 64, STAGE = XA + XW;  // 16-byte units of a stage
    constexpr int FA = BM / 8 / WAVES, FW = BT * KS / WAVES, PER = FA + FW;   // loads of a wave a stage: 1 KiB each
    static_assert(BM / 8 % WAVES == 0 && BT * KS % WAVES == 0, "a stage must divide evenly over the waves");
    static_assert((ST - 1) * PER < 64, "more loads under way than the counter counts");
    static_assert(!SWIGLU || sizeof(TO) == 2, "the activation leaves in bfloat16");
    constexpr int NOUT = SWIGLU ? NTW / 2 : NTW;
    extern __shared__ __align__(16) mbf16x8_t lds[];                     // [ST][STAGE]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave % WM, wn = wave / WM, col = lane & 15, grp = lane >> 4;
    // the row blocks of one block of columns run on one XCD (consecutive block ids go around the eight of them)
    const int id = (int)blockIdx.x, turn = id >> 3;
    const int nb = (turn / mblocks) * 8 + (id & 7), mb = turn % mblocks;
    if (nb >= nblocks) return;
    const int m0 = mb * BM, nks = K / 32, ntiles = N / 16;
    const int s_begin = blockIdx.y * stretches_per_part, s_end = min(nks / KS, s_begin + stretches_per_part);
    C += (size_t)blockIdx.y * part_stride;

    // What this wave brings in.  A: groups of 8 rows, 128 bytes each, 8 lanes a row (lanes next to each other must
    // ask for bytes next to each other: a tenth of the time); a row's eight units of 16 bytes are xor-ed with the
    // row's number and the parity of its group, so that the 16 rows of a read lie in different banks.  W: tiles as
    // they lie.  Rows and tiles beyond the end are read (clamped) and never stored.
    const bf16_t* fa[FA];
    const bf16_t* fw[FW];
#pragma unroll
    for (int i = 0; i < FA; ++i) {
        const int rg = wave * FA + i;
        fa[i] = A + (size_t)min(m0 + rg * 8 + (lane >> 3), M - 1) * lda + ((lane & 7) ^ (lane >> 3) ^ (rg & 1)) * 8;
    }
#pragma unroll
    for (int i = 0; i < FW; ++i) {
        const int f = wave * FW + i, t = f / KS, u = f % KS, w = t / NTW, j = t % NTW;   // k-step u of tile j of the waves w
        const int tile = min((nb * WN + w) * NOUT + j % NOUT, ntiles - 1) + (j >= NOUT ? ntiles : 0);
        fw[i] = W + (((size_t)tile * nks + u) * 64 + lane) * 8;
    }
    auto fetch = [&](int s, int at) {
#pragma unroll
        for (int i = 0; i < FW; ++i)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(fw[i] + (size_t)s * (KS * 512)),
                (__attribute__((address_space(3))) void*)(lds + at + XA + (wave * FW + i) * 64), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < FA; ++i)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(fa[i] + s * (KS * 32)),
                (__attribute__((address_space(3))) void*)(lds + at + (wave * FA + i) * 64), 16, 0, 0);
    };
    const int xat = (wm * MW * 2 + (col >> 3)) * 64 + (col & 7) * 8, xsw = grp ^ (col & 7) ^ (col >> 3);
    const int wat = XA + wn * NTW * KS * 64 + lane;
    auto read = [&](int at, int u, mbf16x8_t (&x)[MW], mbf16x8_t (&w)[NTW]) {
#pragma unroll
        for (int j = 0; j < NTW; ++j) w[j] = lds[at + wat + (j * KS + u) * 64];
#pragma unroll
        for (int i = 0; i < MW; ++i) x[i] = lds[at + xat + i * 128 + (xsw ^ (u * 4))];
    };
    mf32x4_t acc[NTW][MW];
#pragma unroll
    for (int j = 0; j < NTW; ++j)
#pragma unroll
        for (int i = 0; i < MW; ++i) acc[j][i] = mf32x4_t{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const mbf16x8_t (&x)[MW], const mbf16x8_t (&w)[NTW]) {
#pragma unroll
        for (int i = 0; i < MW; ++i)
#pragma unroll
            for (int j = 0; j < NTW; ++j) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j], x[i], acc[j][i], 0, 0, 0);
    };
    // A stage is read in two halves, each asked for ahead of the other half's matrix instructions; between them all waves
    // meet: the stage has been read by all (its place is free for the stage ST further on), and the next one has arrived.
    // (Only the second half's reads have instructions beside them: behind the branch for a last stage the compiled loop waits
    // for all of LDS, so the next stage's first half is in before the second half is multiplied.)
    mbf16x8_t x0[MW], w0[NTW], x1[MW], w1[NTW];
#pragma unroll
    for (int p = 0; p < ST; ++p)
        if (s_begin + p < s_end) fetch(s_begin + p, p * STAGE);
    if (s_begin < s_end) {
        if (s_begin + ST - 1 < s_end) __builtin_amdgcn_s_waitcnt(wait_imm((ST - 1) * PER));
        else __builtin_amdgcn_s_waitcnt(wait_imm(0));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        int at = 0;
        read(at, 0, x0, w0);
        for (int s = s_begin; s < s_end; ++s) {
            __builtin_amdgcn_s_waitcnt(0xc07f);                  // lgkmcnt 0: the first half, asked for a half ago
            read(at, 1, x1, w1);
            multiply(x0, w0);
            const int next = at + STAGE == ST * STAGE ? 0 : at + STAGE;
            if (s + 1 < s_end) {
                asm volatile("" ::: "memory");
                // the loads of the stages after the next one may stay under way (towards the end there are fewer)
                if (s + ST - 1 < s_end) __builtin_amdgcn_s_waitcnt(wait_imm((ST - 2) * PER));
                else __builtin_amdgcn_s_waitcnt(wait_imm(0));
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                if (s + ST < s_end) fetch(s + ST, at);
                read(next, 0, x0, w0);
            }
            multiply(x1, w1);
            at = next;
        }
    }
    // acc[j][i][e] = C[m0 + (wm * MW + i) * 16 + col][tile j * 16 + grp * 4 + e]
#pragma unroll
    for (int j = 0; j < NOUT; ++j) {
        const int tile = (nb * WN + wn) * NOUT + j;
        if (tile >= ntiles) break;
        const int n = tile * 16 + grp * 4;
#pragma unroll
        for (int i = 0; i < MW; ++i) {
            const int m = m0 + (wm * MW + i) * 16 + col;
            if (m >= M) continue;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = acc[j][i][e];
                if (SWIGLU) v[e] = v[e] / (1.f + __expf(-v[e])) * acc[NOUT + j][i][e];
            }
            VecLoad<4>::st(C + (size_t)m * ldc + n, v);
        }
    }
}

template <int WM, int WN, int MW, int NTW, int ST, bool SWIGLU, typename TO>
int launch_mid(const bf16_t* A, int lda, const bf16_t* W, TO* C, int ldc, int M, int N, int K, int parts, size_t part_stride,
               hipStream_t stream) {
    constexpr int BM = WM * MW * 16, NOUT = SWIGLU ? NTW / 2 : NTW;
    constexpr size_t lds = (size_t)ST * (BM * KS * 4 + WN * NTW * KS * 64) * 16;
    static_assert(lds > 64 * 1024 && lds <= 160 * 1024, "more LDS than a kernel may take unasked, no more than there is");
    auto kernel = gemm_mid_kernel<WM, WN, MW, NTW, ST, SWIGLU, TO>;
    {
        static std::mutex mu;
        static bool asked[64] = {};
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        RI_REQUIRE(e == hipSuccess && dev >= 0 && dev < 64, "ri_gemm_mid: no current device: %s", hipGetErrorString(e));
        std::lock_guard<std::mutex> lock(mu);
        if (!asked[dev]) {
            e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            RI_REQUIRE(e == hipSuccess, "ri_gemm_mid: %zu bytes of LDS refused: %s", lds, hipGetErrorString(e));
            asked[dev] = true;
        }
    }
    const int mblocks = (M + BM - 1) / BM, nblocks = (N / 16 + WN * NOUT - 1) / (WN * NOUT);
    const int s_all = K / 32 / KS;
    kernel<<<dim3((nblocks + 7) / 8 * 8 * mblocks, parts), WM * WN * 64, lds, stream>>>(
        A, lda, W, C, ldc, M, N, K, mblocks, nblocks, (s_all + parts - 1) / parts, part_stride);
    return 0;
}

template <bool SWIGLU, typename TO>
int dispatch_mid(const bf16_t* A, int lda, const bf16_t* W, TO* C, int ldc, int M, int N, int K, int wide, int parts,
                 size_t part_stride, hipStream_t stream) {
    // blocks of 128 rows and 8 weight tiles (eight waves, a compute unit's LDS) or 4 (four waves, two blocks a unit)
    if (wide) return launch_mid<4, 2, 2, 4, 4, SWIGLU, TO>(A, lda, W, C, ldc, M, N, K, parts, part_stride, stream);
    return launch_mid<2, 2, 4, 2, 3, SWIGLU, TO>(A, lda, W, C, ldc, M, N, K, parts, part_stride, stream);
}

}  // namespace

// What a product in `parts` slices and the kernel after it take, in us, fitted to 860 measured triples of sizes, slices and
// widths (16 and 9 weights from 768 x 768 to 12288 x 4096, 65 to 2,048 rows, replayed in a graph; 5 % off for the norm, 11 % for
// the rotation): a stretch of 64 values of K takes a wide block 0.48, a narrow one 0.39, or two narrow ones on a unit 0.60; the
// chip does 256 wide blocks at once, or 512 narrow ones, as long as no XCD gets more than its share, which `across` counts (the
// blocks of one block of columns run on one XCD: 20 of those leave four XCDs with three, so 384 rows of 2560 x 2560 in
// four slices took two rounds, 29 us, 21 in the library); then the sums: c0 a result and c1 a result and slice,
// and what the rotation's kernel takes to read a token's row, slice after slice.
static float mid_time(int M, int N, int K, int parts, int wide, int rotated) {
    const int bt = wide ? 8 : 4;
    const long long across = ((N / 16 + bt - 1) / bt + 7) / 8 * 8, blocks = across * ((M + 127) / 128) * parts;
    const int stretches = (K / 64 + parts - 1) / parts;
    // (slices that make a second round never paid: 4096 x 14336 with 300 rows, 2 slices 66 us, 4 76, 8 74)
    if (parts > 1 && blocks > (wide ? 256 : 512)) return 1e30f;
    const float stretch = wide ? 0.48f * ((blocks + 255) / 256) : blocks <= 256 ? 0.39f : 0.60f * ((blocks + 511) / 512);
    const float results = 1e-6f * M * N;
    return stretch * stretches + (rotated ? results * (3.07f + 1.02f * parts) + 0.38e-3f * N * parts : results * (1.55f + 1.57f * parts));
}

// Whether and how gemm_mid takes a product of M rows, N columns (SwiGLU: of each half) and K inner values: the
// slices of K (0: it does not) and whether a block owns 8 weight tiles or 4.  It takes what leaves the GEMM
// library's tiles of 128 x 128 on at most half of the 256 compute units (with 192 such tiles the library is as fast, and
// faster beyond), in the slices, of at least 256 values of K, that take the least time.  `rotated`: the kernel that
// rotates adds the sums, any number of slices up to 8; else the norm does, a power of two.
//
// A SwiGLU product, whose sums cannot be divided, is taken where its blocks fit the units once, narrow ones if those do.
// us, weights from memory, library with its activation kernel / narrow / wide: 2 x 8192 x 2048, 128 rows (128 wide blocks) 30 / 21 / 25;
// 2 x 8704 x 4096, 128 rows (136) 46 / 54 / 43; 2 x 11008 x 4096, 128 rows (172) 49 / 57 / 46; 2 x 5632 x 4096, 256 rows (176) 52 / 51 / 41;
// 2 x 14336 x 4096, 128 rows (224) 58 / 60 / 51; 2 x 9472 x 2560, 256 rows (296) 51 / 54 / 54; 2 x 8192 x 2048, 320 rows (384)
// 34 / 41 / 41, 512 rows (512) 42 / 54 / 44.
extern "C" int ri_gemm_mid_plan(int M, int N, int K, int swiglu, int rotated, int* parts_out, int* wide_out) {
    RI_REQUIRE(parts_out && wide_out && M > 0 && N > 0 && K > 0, "ri_gemm_mid_plan: bad arguments");
    *parts_out = 0;
    *wide_out = 1;
    if (M <= 64 || N % 16 || K % 64) return 0;
    const long long mblocks = (M + 127) / 128;
    if (swiglu) {
        auto blocks = [&](int tiles) { return ((N / 16 + tiles - 1) / tiles + 7) / 8 * 8 * mblocks; };
        if (blocks(4) > 256) return 0;
        *wide_out = blocks(2) > 256;
        *parts_out = 1;
        return 0;
    }
    if (mblocks * ((N / 16 + 7) / 8) > 128) return 0;
    float least = 0.f;
    for (int p = 1; p <= 8; p = rotated ? p + 1 : 2 * p) {
        if (p > 1 && K / 64 / p < 4) break;
        for (int wide = 0; wide < 2; ++wide) {
            const float t = mid_time(M, N, K, p, wide, rotated);
            if (*parts_out == 0 || t < least) { least = t; *parts_out = p; *wide_out = wide; }
        }
    }
    return 0;
}

// W: the copy in tile order.  swiglu != 0: W is [2N, K] (gate rows, then up rows), C [M, ldc] bfloat16, parts 1.
// Else C is a float32 stack [parts][M][ldc] (part_stride elements apart) of partial sums over slices of K.
extern "C" int ri_gemm_mid(const void* A, int lda, const void* W, void* C, int ldc, int M, int N, int K, int swiglu,
                           int parts, int wide, long long part_stride, hipStream_t stream) {
    RI_REQUIRE(M >= 1 && N > 0 && N % 16 == 0 && K > 0 && K % 64 == 0, "ri_gemm_mid: needs N %% 16 == 0 and K %% 64 == 0 (M=%d N=%d K=%d)", M, N, K);
    RI_REQUIRE(lda >= K && lda % 8 == 0 && ldc >= N && ldc % 4 == 0, "ri_gemm_mid: bad leading dimensions");
    RI_REQUIRE(A && W && C && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0 && (uintptr_t)C % 16 == 0, "ri_gemm_mid: null or unaligned pointer");
    RI_REQUIRE(parts >= 1 && parts <= 64 && (!swiglu || parts == 1), "ri_gemm_mid: parts=%d", parts);
    RI_REQUIRE(parts == 1 || (part_stride >= (long long)M * ldc && part_stride % 4 == 0), "ri_gemm_mid: the slices overlap");
    RI_REQUIRE((long long)((M + 127) / 128) * (N / 16 + 7) < (1ll << 31), "ri_gemm_mid: M=%d N=%d exceed the grid limit", M, N);
    const size_t ps = parts > 1 ? (size_t)part_stride : 0;
    int rc;
    if (swiglu) rc = dispatch_mid<true, bf16_t>((const bf16_t*)A, lda, (const bf16_t*)W, (bf16_t*)C, ldc, M, N, K, wide, 1, 0, stream);
    else rc = dispatch_mid<false, float>((const bf16_t*)A, lda, (const bf16_t*)W, (float*)C, ldc, M, N, K, wide, parts, ps, stream);
    if (rc) return rc;
    RI_LAUNCHED("ri_gemm_mid");
    return 0;
}
