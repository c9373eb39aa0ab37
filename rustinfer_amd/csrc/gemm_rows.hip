// C[M, N] = A[M, K] . W[N, K]^T for 8 to 64 rows of bfloat16 against weights in tile order
// ([N/16][K/32][64 lanes][8], see gemm.hip), with the activations shared through LDS.
//
// From 17 rows on a wave of the few-row kernel (gemm.hip) asks for as many bytes of
// activations as of weights, and the product takes as long as if both came from memory; with fewer it is the kernel's registers that limit what
// is under way.  Here
// the waves of a group work on the same 64 values of K at a time: the group brings that stretch of all (up to 64) rows into LDS once,
// and each of its waves the stretch of weight tiles of its own beside it, with loads that write LDS directly, into a ring of
// two to four stages, in the order in which the matrix instructions read them.  What is asked of memory is then the weights, once, and
// one copy of the activations a block, and nothing but a wave's own counter of loads and one barrier a stage stands between
// them and the products.  (Through registers a stretch ahead, the compiled loop waited for every load before it asked for the next stretch;
// with those waits gone, copies of the loads' registers still waited for most of them.)
//
// A block owns 2 or 4 waves' NT tiles of 16 columns (SWIGLU: as many of the gate half and of the up half of
// a stacked [2N, K] matrix, and writes silu(gate) * up).  Products with few columns are also
// split over K between blocks (blockIdx.y), each leaving 32-bit partial sums in its own slice of
// C, which the norm that follows adds up, and a block holds two or four groups of waves, which split its share of K between them
// through rings of their own.  N % 16 == 0, K % 32 == 0.
//
// What bounds it: bytes in flight, and the launch.  Measured, us, 20 / 40 / 64 rows, through registers / now, and a kernel that only reads as much: gate/up
// 2 x 8192 x 2048 16.4 17.1 18.1 / 14.3 15.0 16.8 (11.3), 2 x 8192 x 3072 22.6 24.2 25.5 / 19.7 21.1 22.9 (16.2), 2 x 14336 x 4096 48 49 52 / 45 47 49 (35.6); q/k/v with
// rotation 5120 x 3072 13.3 15.8 19.1 / 11.3 13.8 16.4 (6.2); in slices 2048 x 8192 11.0 11.0 12.1 / 8.5 9.0 9.9 (6.5), 3072 x 3072 7.7 8.3 9.4 / 6.1 7.1 8.2 (4.3); whole
// 128256 x 3072 137 144 154 / 134 141 149 (116).  Up to 16 rows, the few-row kernel / this one at 8, 16 rows: in slices 2048 x 8192 9.0 9.1 / 7.7 7.8 (6.5),
// 3072 x 8192 14.1 12.6 / 11.0 11.1 (8.9), 5120 x 5120 13.7 14.0 / 11.3 12.1 (9.2); whole 16384 x 2048 14.9 18.0 / 13.7 13.8 (11.3).
// Whole products of fewer columns at 17, 33, 64 rows: 8192 x 2048 10.1 19.1 20.6 / 8.9 9.8 11.1, 12288 x 4096 26 36 36 / 24 25 26.
#include "common.h"
#include <mutex>

typedef __bf16 rbf16x8_t __attribute__((ext_vector_type(8)));
typedef float rf32x4_t __attribute__((ext_vector_type(4)));

namespace {

constexpr int KS = 2;                     // k-steps of 32 in a stretch: 128 bytes of a row

// s_waitcnt: at most n loads under way, and nothing asked of LDS: a stage is written over behind the barrier only when what was read of it has arrived
constexpr int loads_imm(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4); }

struct Store4 {
    static __device__ __forceinline__ void st(float* p, const float* v) {
        *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
    }
    static __device__ __forceinline__ void st(bf16_t* p, const float* v) {
        uint2 t;
        t.x = (uint32_t)f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16);
        t.y = (uint32_t)f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16);
        *reinterpret_cast<uint2*>(p) = t;
    }
};

// ROPE: the product is the fused q/k/v projection of a step's tokens, with the weight's rows permuted
// within each head as for the few-row kernel (gemm.hip, ri_qkv_rope_row_order): a tile holds 8
// features of the first half of a head and their 8 partners, the partner of a lane's value sits in
// lane ^ 32.  The epilogue rotates q and k by the token's position (32-bit, one rounding), writes
// k and v into the token's cache page and only q to C.
struct RowsRope {
    const float* cos_t; const float* sin_t;        // [positions][hd / 2]
    const int* positions; const int* row_of_token; // per token (row of A)
    const int* table; int max_blocks;              // block table [rows][max_blocks]
    bf16_t* kc; bf16_t* vc;                        // k [pages][Hkv][page][hd], v [pages][Hkv][hd][page]
    int H, Hkv, hd, page;
};

// KG groups of WAVES waves share a block: each group takes its own share of the block's stretches, through a ring of its own of ST stages, and the
// groups' sums meet in LDS at the end.
template <int MT, int NT, bool SWIGLU, typename TO, int WAVES, int KG, int ST, bool ROPE = false>
__global__ __launch_bounds__(WAVES * KG * 64) void gemm_rows_lds_kernel(
        const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W,
        TO* __restrict__ C, int ldc, int M, int N, int K, int stretches_per_block, size_t part_stride,
        RowsRope rp) {
    static_assert(!ROPE || (NT == 1 && !SWIGLU && sizeof(TO) == 2), "the rotation goes with one bfloat16 tile a wave");
    constexpr int NW = SWIGLU ? 2 * NT : NT;
    constexpr int XPIECES = MT * 2, FX = (XPIECES + WAVES - 1) / WAVES;        // kilobytes of the rows in a stage: eight rows each; a wave's
    constexpr int XA = XPIECES * 64, STAGE = XA + WAVES * NW * KS * 64;        // in units of 16 bytes
    constexpr int PER = FX + NW * KS;                                          // loads of a wave a stage
    static_assert((ST - 1) * PER < 64, "more loads under way than the counter counts");
    extern __shared__ __align__(16) rbf16x8_t xs_all[];     // [KG][ST][STAGE]
    // a wave's group and its number in it, the same in all its lanes
    const int all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kg = all / WAVES, wave = all % WAVES;
    rbf16x8_t* xs = xs_all + kg * ST * STAGE;
    const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
    const int ntiles = N / 16, nks_all = K / 32;
    const int s_all = (nks_all + KS - 1) / KS;
    const int b_begin = blockIdx.y * stretches_per_block;
    const int b_end = min(s_all, b_begin + stretches_per_block);
    const int span = (max(b_end - b_begin, 0) + KG - 1) / KG;      // stretches of a group; the same for all
    const int s_begin = b_begin + kg * span;
    const int s_end = min(b_end, s_begin + span);
    C += (size_t)blockIdx.y * part_stride;

    // What this wave brings in.  Rows: eight a load, 128 bytes each, eight lanes a row; a row's eight units of 16 bytes are xor-ed
    // with the row's number and the parity of its eight, so that the 16 rows of a read lie in different banks.  Weights: its own
    // tiles, as they lie.  Rows and tiles beyond the end are read (clamped) and never stored; of an odd last step, the step before it is
    // read again and not multiplied.
    size_t fx[FX];
#pragma unroll
    for (int i = 0; i < FX; ++i) {
        const int p = min(wave * FX + i, XPIECES - 1);
        fx[i] = (size_t)min(p * 8 + (lane >> 3), M - 1) * lda + ((lane & 7) ^ (lane >> 3) ^ (p & 1)) * 8;
    }
    const bf16_t* wp[NW];
#pragma unroll
    for (int a = 0; a < NW; ++a) {
        const int tile = min(((int)blockIdx.x * WAVES + wave) * NT + (a % NT), ntiles - 1) + (a >= NT ? ntiles : 0);
        wp[a] = W + ((size_t)tile * nks_all * 64 + lane) * 8;
    }
    auto fetch = [&](int s, int at) {
#pragma unroll
        for (int u = 0; u < KS; ++u)
#pragma unroll
            for (int a = 0; a < NW; ++a)
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(wp[a] + (size_t)min(s * KS + u, nks_all - 1) * 512),
                    (__attribute__((address_space(3))) void*)(xs + at + XA + ((wave * NW + a) * KS + u) * 64), 16, 0, 2);
        const bool odd = (s + 1) * KS > nks_all;
#pragma unroll
        for (int i = 0; i < FX; ++i) {
            const int p = min(wave * FX + i, XPIECES - 1);
            const size_t from = fx[i] - (odd && (((lane & 7) ^ (lane >> 3) ^ (p & 1)) & 4) ? 32 : 0);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(A + (size_t)s * (KS * 32) + from),
                (__attribute__((address_space(3))) void*)(xs + at + p * 64), 16, 0, 0);
        }
    };
    rf32x4_t acc[NW][MT];
#pragma unroll
    for (int a = 0; a < NW; ++a)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[a][mt] = rf32x4_t{0.f, 0.f, 0.f, 0.f};
    const int xat = (col >> 3) * 64 + (col & 7) * 8, xsw = grp ^ (col & 7) ^ (col >> 3);
    const int wat = XA + wave * NW * KS * 64 + lane;
    auto multiply = [&](int at, int u) {
        rbf16x8_t xf[MT], wf[NW];
#pragma unroll
        for (int a = 0; a < NW; ++a) wf[a] = xs[at + wat + (a * KS + u) * 64];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) xf[mt] = xs[at + xat + mt * 128 + (xsw ^ (u * 4))];
#pragma unroll
        for (int a = 0; a < NW; ++a)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                acc[a][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[a], xf[mt], acc[a][mt], 0, 0, 0);
    };
    // What the rotation needs of each token is asked for at the start, its row and position ahead of the first stages, its page, cosines and sines behind
    // them: a chain of small loads at the end of a short kernel would cost microseconds.
    int rp_section = 0, rp_head = 0, rp_j = 0;
    int rp_b[ROPE ? MT : 1], rp_blk[ROPE ? MT : 1], rp_slot[ROPE ? MT : 1];
    float4 rp_c[ROPE ? MT : 1], rp_s[ROPE ? MT : 1];
    if constexpr (ROPE) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int m = mt * 16 + col;
            rp_b[mt] = -1; rp_slot[mt] = 0;
            if (kg == 0 && m < M) { rp_b[mt] = rp.row_of_token[m]; rp_slot[mt] = rp.positions[m]; }
        }
    }
#pragma unroll
    for (int p = 0; p < ST - 1; ++p)
        if (s_begin + p < s_end) fetch(s_begin + p, p * STAGE);
    if constexpr (ROPE) {
        const int hd = rp.hd, half = hd >> 1, q_dim = rp.H * hd, kv_dim = rp.Hkv * hd;
        const int n0 = min(((int)blockIdx.x * WAVES + wave), ntiles - 1) * 16;
        rp_section = n0 < q_dim ? 0 : (n0 < q_dim + kv_dim ? 1 : 2);                     // q, k, v
        const int within = n0 - (rp_section == 0 ? 0 : (rp_section == 1 ? q_dim : q_dim + kv_dim));
        rp_head = within / hd;
        rp_j = (within % hd) >> 4;                                                       // the tile is tile j of its head
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int b = rp_b[mt], pos = rp_slot[mt];
            rp_blk[mt] = -1;
            rp_slot[mt] = pos % rp.page;
            rp_c[mt] = make_float4(1.f, 1.f, 1.f, 1.f);
            rp_s[mt] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (b >= 0) {
                if (rp_section != 0) rp_blk[mt] = rp.table[(size_t)b * rp.max_blocks + pos / rp.page];
                if (rp_section != 2) {
                    // this lane's four values are features 8 j + (grp & 1) 4 + i of a half
                    const size_t at = (size_t)pos * half + 8 * rp_j + (grp & 1) * 4;
                    rp_c[mt] = *reinterpret_cast<const float4*>(rp.cos_t + at);
                    rp_s[mt] = *reinterpret_cast<const float4*>(rp.sin_t + at);
                }
            }
        }
    }

    // A stage: this wave's loads of it have arrived, then, behind the barrier, everyone's, and all have read the stage before it, into whose
    // place the next loads go.  Every wave passes the same barriers, with or without a stretch of its own left.
    int at = 0;
    for (int s = s_begin; s < s_begin + span; ++s) {
        // (what the rotation asked for behind the first stages counts as under way: fewer may, for one stage)
        if (s + ST - 2 < s_end) __builtin_amdgcn_s_waitcnt(loads_imm((ST - 2) * PER));
        else __builtin_amdgcn_s_waitcnt(loads_imm(0));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (s + ST - 1 < s_end) fetch(s + ST - 1, at == 0 ? (ST - 1) * STAGE : at - STAGE);
        if (s < s_end) {
            multiply(at, 0);
            if (s * KS + 1 < nks_all) multiply(at, 1);
        }
        at = at + STAGE == ST * STAGE ? 0 : at + STAGE;
    }
    if (KG > 1) __syncthreads();
    if (KG > 1) {
        // the other groups' sums, through the LDS the stretches have left: [group - 1][wave][a][mt][lane]
        rf32x4_t* red = reinterpret_cast<rf32x4_t*>(xs_all);
        if (kg > 0) {
#pragma unroll
            for (int a = 0; a < NW; ++a)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    red[((((kg - 1) * WAVES + wave) * NW + a) * MT + mt) * 64 + lane] = acc[a][mt];
        }
        __syncthreads();
        if (kg > 0) return;
#pragma unroll
        for (int g = 1; g < KG; ++g)
#pragma unroll
            for (int a = 0; a < NW; ++a)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const rf32x4_t o = red[((((g - 1) * WAVES + wave) * NW + a) * MT + mt) * 64 + lane];
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[a][mt][i] += o[i];
                }
    }

    // acc[a][mt][i] = C[m = mt * 16 + col][n = tile(a) * 16 + grp * 4 + i]
    if constexpr (ROPE) {
        if ((int)blockIdx.x * WAVES + wave >= ntiles) return;
        const int hd = rp.hd, half = hd >> 1;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int m = mt * 16 + col;
            const int b = rp_b[mt], blk = rp_blk[mt], slot = rp_slot[mt];
            const float cs[4] = {rp_c[mt].x, rp_c[mt].y, rp_c[mt].z, rp_c[mt].w};
            const float sn[4] = {rp_s[mt].x, rp_s[mt].y, rp_s[mt].z, rp_s[mt].w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = grp * 4 + i;                           // row of the tile: r < 8 first half, else partner
                const float v = acc[0][mt][i];
                const float other = __shfl_xor(v, 32, 64);           // row r ^ 8, same token
                const int fi = 8 * rp_j + (r & 7);                   // index within the half
                const int d = r < 8 ? fi : half + fi;                // feature within the head
                if (b < 0) continue;                                 // padding token or beyond M
                if (rp_section == 2) {
                    if (blk >= 0) rp.vc[((size_t)blk * rp.Hkv + rp_head) * rp.page * hd + (size_t)d * rp.page + slot] = f32_to_bf16(v);
                    continue;
                }
                const float res = r < 8 ? v * cs[i] - other * sn[i] : other * sn[i] + v * cs[i];
                if (rp_section == 0) st_f32(C + (size_t)m * ldc + rp_head * hd + d, res);
                else if (blk >= 0) rp.kc[((size_t)blk * rp.Hkv + rp_head) * rp.page * hd + (size_t)slot * hd + d] = f32_to_bf16(res);
            }
        }
        return;
    }
#pragma unroll
    for (int a = 0; a < NT; ++a) {
        const int tile = ((int)blockIdx.x * WAVES + wave) * NT + a;
        if (tile >= ntiles) break;
        const int n = tile * 16 + grp * 4;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int m = mt * 16 + col;
            if (m >= M) continue;
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[i] = acc[a][mt][i];
                if (SWIGLU) v[i] = v[i] / (1.f + __expf(-v[i])) * acc[NT + a][mt][i];
            }
            TO* dst = C + (size_t)m * ldc + n;
            if ((ldc & 3) == 0 && ((uintptr_t)C & 15) == 0) {
                Store4::st(dst, v);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) st_f32(dst + i, v[i]);
            }
        }
    }
}

// Stages of a ring: what fits half a compute unit's LDS with one group, a whole one's with more, two to four.
constexpr int ring(int stage_units, int kg, int most) {
    const int fit = (kg == 1 ? 80 : 152) * 64 / (stage_units * kg);
    return fit < 2 ? 2 : fit > most ? most : fit;
}

template <int MT, int NT, bool SWIGLU, typename TO, int KG>
int launch_rows_groups(const bf16_t* A, int lda, const bf16_t* W, TO* C, int ldc, int M, int N, int K,
                       int parts, size_t part_stride, hipStream_t stream) {
    // Four waves a group; `four groups`: of two waves, so that a block owns half the columns.  With two weight tiles a wave (SwiGLU) four groups leave
    // room for two stages, which is not enough under way: two groups of four stages (8192 x 3072, 40 rows, four groups of two 24.7 us, two of four 21.1).
    constexpr int waves = KG == 4 ? 2 : 4, groups = KG == 4 && SWIGLU ? 2 : KG;
    constexpr int stage = MT * 128 + waves * (SWIGLU ? 2 * NT : NT) * KS * 64, ST = ring(stage, groups, KG == 4 && SWIGLU ? 4 : 3);
    constexpr size_t lds = (size_t)groups * ST * stage * sizeof(rbf16x8_t);
    static_assert(lds <= 160 * 1024, "a compute unit's LDS");
    auto kernel = gemm_rows_lds_kernel<MT, NT, SWIGLU, TO, waves, groups, ST>;
    if (lds > 64 * 1024) {          // beyond what a kernel may take unasked: ask once a device
        static std::mutex mu;
        static bool asked[64] = {};
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        RI_REQUIRE(e == hipSuccess && dev >= 0 && dev < 64, "ri_gemm_rows_bf16: no current device: %s", hipGetErrorString(e));
        std::lock_guard<std::mutex> lock(mu);
        if (!asked[dev]) {
            e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            RI_REQUIRE(e == hipSuccess, "ri_gemm_rows_bf16: %zu bytes of LDS refused: %s", lds, hipGetErrorString(e));
            asked[dev] = true;
        }
    }
    const int s_all = (K / 32 + KS - 1) / KS;
    const int per = (s_all + parts - 1) / parts;
    const int blocks = (N / 16 + waves * NT - 1) / (waves * NT);
    kernel<<<dim3(blocks, parts), waves * groups * 64, lds, stream>>>(A, lda, W, C, ldc, M, N, K, per, part_stride, RowsRope{});
    return 0;
}

template <int MT, int NT, bool SWIGLU, typename TO>
int launch_rows(const bf16_t* A, int lda, const bf16_t* W, TO* C, int ldc, int M, int N, int K,
                int parts, size_t part_stride, int groups, hipStream_t stream) {
    if (groups == 2) return launch_rows_groups<MT, NT, SWIGLU, TO, 2>(A, lda, W, C, ldc, M, N, K, parts, part_stride, stream);
    if (groups == 4) return launch_rows_groups<MT, NT, SWIGLU, TO, 4>(A, lda, W, C, ldc, M, N, K, parts, part_stride, stream);
    return launch_rows_groups<MT, NT, SWIGLU, TO, 1>(A, lda, W, C, ldc, M, N, K, parts, part_stride, stream);
}

template <int NT, bool SWIGLU, typename TO>
int dispatch_rows(const bf16_t* A, int lda, const bf16_t* W, TO* C, int ldc, int M, int N, int K,
                  int parts, size_t part_stride, int groups, hipStream_t stream) {
    if (M <= 16) return launch_rows<1, NT, SWIGLU, TO>(A, lda, W, C, ldc, M, N, K, parts, part_stride, groups, stream);
    if (M <= 32) return launch_rows<2, NT, SWIGLU, TO>(A, lda, W, C, ldc, M, N, K, parts, part_stride, groups, stream);
    if (M <= 48) return launch_rows<3, NT, SWIGLU, TO>(A, lda, W, C, ldc, M, N, K, parts, part_stride, groups, stream);
    return launch_rows<4, NT, SWIGLU, TO>(A, lda, W, C, ldc, M, N, K, parts, part_stride, groups, stream);
}

// The fused q/k/v projection with rotation: four groups of two waves a block (32 columns) or two
// groups of four (64 columns), see launch_rows_groups.
template <int MT, int KG>
int launch_rows_rope(const bf16_t* A, int lda, const bf16_t* W, bf16_t* C, int ldc, int M, int N, int K,
                     const RowsRope& rp, hipStream_t stream) {
    static_assert(KG == 2 || KG == 4, "two or four groups");
    constexpr int waves = KG == 4 ? 2 : 4, stage = MT * 128 + waves * KS * 64, ST = ring(stage, KG, 3);
    constexpr size_t lds = (size_t)KG * ST * stage * sizeof(rbf16x8_t);
    static_assert(lds <= 160 * 1024, "a compute unit's LDS");
    auto kernel = gemm_rows_lds_kernel<MT, 1, false, bf16_t, waves, KG, ST, true>;
    if (lds > 64 * 1024) {
        static std::mutex mu;
        static bool asked[64] = {};
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        RI_REQUIRE(e == hipSuccess && dev >= 0 && dev < 64, "ri_gemm_rows_qkv_rope: no current device: %s", hipGetErrorString(e));
        std::lock_guard<std::mutex> lock(mu);
        if (!asked[dev]) {
            e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            RI_REQUIRE(e == hipSuccess, "ri_gemm_rows_qkv_rope: %zu bytes of LDS refused: %s", lds, hipGetErrorString(e));
            asked[dev] = true;
        }
    }
    const int s_all = (K / 32 + KS - 1) / KS;
    const int blocks = (N / 16 + waves - 1) / waves;
    kernel<<<dim3(blocks, 1), waves * KG * 64, lds, stream>>>(A, lda, W, C, ldc, M, N, K, s_all, 0, rp);
    return 0;
}

template <int MT>
int launch_rows_rope_groups(const bf16_t* A, int lda, const bf16_t* W, bf16_t* C, int ldc, int M, int N, int K,
                            int groups, const RowsRope& rp, hipStream_t stream) {
    if (groups == 2) return launch_rows_rope<MT, 2>(A, lda, W, C, ldc, M, N, K, rp, stream);
    return launch_rows_rope<MT, 4>(A, lda, W, C, ldc, M, N, K, rp, stream);
}

}  // namespace

// Slices of K, and wave groups a block, for a product of M rows, N columns and K inner values whose partial sums a norm adds up: blocks enough to
// fill the chip twice, at most 8 slices (16 of 2048 x 8192 take less here and cost the norm more), then groups where that fills the units better with as many
// slices or fewer.  Up to 16 rows and for 16 to 80 blocks of 64 columns: eight slices, in four groups up to 32 blocks (and of 64 with rows of 8,192 values or more), in two for
// 56 to 64 with shorter rows, else in one, whose blocks all run at once; parts 1 elsewhere, where the few-row kernel is as fast.  16 rows, us, few-row / eight slices in 1, 2, 4 groups:
// 1088 x 8192 8.0 / 7.8 6.4 6.6, 1536 x 8960 9.6 / 10.4 8.0 8.2, 1984 x 4096 6.5 / 5.6 5.4 5.3, 2048 x 8192 9.3 / 9.1 8.5 7.9; 2560 x 9728 12.9 / 11.3 12.2 11.5, 3328 x 4096 9.8 /
// 7.2 7.3 8.0; 3584 x 3584 9.2 / 7.0 6.9 8.0, 3584 x 7168 16.1 / 10.9 11.4 12.2, 3840 x 5120 12.2 / 8.6 8.8 9.9, 4096 x 4096 8.6 / 9.6 8.4 9.1.  us, few-row / this at 9 to 16 rows: 2048 x 2048 4.6
// / 4.1, 2048 x 8192 8.8 / 7.7, 3072 x 8192 12.5 / 11.0, 4096 x 4096 8.7 / 8.5, 4096 x 14336 22.2 / 20.9, 5120 x 5120 14.0 / 12.1, 5120 x 13824 29.4 / 27.5.  With more: a block of two groups has a unit to itself (two share it up to 32 rows), three of one group share one
// (four up to 32 rows), and one of four groups, of half the columns, has one to itself.  Measured, us (slices/groups), at 20, 32, 48, 64 rows: 2048 x 2048
// 4/4 4.5 4.7 5.2 5.6, 8/1 4.9 5.2 5.7 6.0; 1024 x 3072 8/4 4.1 4.3 4.8 5.3, 8/1 4.7 5.0 5.5 5.9; 2048 x 8192 8/2 8.5 8.7 9.2 9.9, 4/4 9.9 10.4 11.2 11.7, 8/1 9.0 9.1
// 9.8 10.6; 3072 x 8192 4/2 11.6 12.0 13.2 14.3, 8/1 11.1 11.7 13.7 15.4; 4096 x 4096 8/2 9.0 9.5 - -, 4/2 9.9 10.2 10.8 11.5, 8/1 9.6 10.1 10.8 11.8; 4096 x 14336 8/2
// 22.0 22.9 27.3 29.7, 4/2 21.2 21.9 23.9 25.4, 8/1 21.5 21.7 24.4 26.5; 5120 x 13824 8/1 28.1 29.5 33.1 35.8, 4/1 29.4 31.6 36.7 40.5; 5120 x 5120 4/1 12.7 13.9 16.8
// 18.1, 8/1 12.5 13.7 15.8 17.3 (and the norm's slices); 8192 x 8192 4/2 28.1 26.7 30.1 31.7, 4/1 29.0 27.8 26.3 28.3.  (Through registers, with the plan of then: 2048 x 2048
// 5.0 5.3 6.4 6.9, 2048 x 8192 11.1 11.3 11.2 12.1, 3072 x 8192 12.5 13.0 14.0 15.6, 4096 x 4096 10.1 10.5 12.2 13.0, 4096 x 14336 22.8 23.2 24.6 26.4.)
extern "C" int ri_gemm_rows_plan(int M, int N, int K, int nt, int* parts_out, int* groups_out) {
    RI_REQUIRE(parts_out && groups_out && N > 0 && K > 0 && (nt == 1 || nt == 2), "ri_gemm_rows_plan: bad arguments");
    const int blocks = (N / 16 + 4 * nt - 1) / (4 * nt), stretches = (K + 63) / 64;
    int parts = 1, groups = 1;
    if (M <= 16) {
        const bool one_round = blocks >= 56 && blocks <= 64 && K < 8192;
        *parts_out = *groups_out = 1;
        if (blocks < 16 || blocks > 80 || stretches < 8) return 0;
        parts = 8;
        groups = one_round ? 2 : blocks <= 32 || (blocks % 32 == 0 && K >= 8192) ? 4 : 1;
        while (groups > 1 && stretches < parts * groups) groups /= 2;
        *parts_out = parts;
        *groups_out = groups;
        return 0;
    }
    while (parts < 8 && blocks * parts < 512 && stretches / (parts * 8) >= 1) parts *= 2;
    // with more than 32 rows no more blocks than the chip holds at once (a long K: three a unit; the norm adds the slices of a short one)
    if (M > 32 && parts > 1 && blocks * parts > (K >= 8192 ? 768 : 512)) parts /= 2;
    if (blocks <= 32 && K <= 4096) {
        parts = blocks <= 16 ? 8 : 4;
        groups = 4;
    } else if (M <= 32) {
        if (blocks * parts <= 256 || (blocks * parts > 460 && blocks * parts <= 512 && K <= 8192)) groups = 2;
    } else if (parts == 8) {
        if (blocks * 8 <= 256) groups = 2;
        else if (blocks * 4 < 256 || (blocks * 4 == 256 && K <= 4096)) { parts = 4; groups = 2; }
    }
    while (parts * groups > 1 && stretches < parts * groups) (groups > 1 ? groups : parts) /= 2;
    *parts_out = parts;
    *groups_out = groups;
    return 0;
}

// W: the copy in tile order.  swiglu != 0: W is [2N, K] (gate rows, then up rows), C bfloat16.
// parts > 1: C is a float32 stack [parts][M][ldc] (part_stride elements apart) of partial sums.
// nt: tiles of 16 columns a wave owns (1 or 2).  groups: 1, or 2 for blocks of eight waves whose
// halves split the block's share of K between them, or 4 for blocks of four pairs of waves that do
// (half the columns a block, so twice the blocks).
extern "C" int ri_gemm_rows_bf16(const void* A, int lda, const void* W, void* C, int ldc, int M, int N, int K,
                                 int out_dtype, int swiglu, int parts, long long part_stride, int nt, int groups,
                                 hipStream_t stream) {
    RI_REQUIRE(groups == 1 || groups == 2 || groups == 4, "ri_gemm_rows_bf16: groups=%d not 1, 2 or 4", groups);
    RI_REQUIRE(M >= 1 && M <= 64, "ri_gemm_rows_bf16: M=%d not in [1, 64]", M);
    RI_REQUIRE(N > 0 && N % 16 == 0 && K > 0 && K % 32 == 0, "ri_gemm_rows_bf16: needs N %% 16 == 0 and K %% 32 == 0 (N=%d K=%d)", N, K);
    RI_REQUIRE(lda >= K && lda % 8 == 0 && ldc >= N, "ri_gemm_rows_bf16: bad leading dimensions");
    RI_REQUIRE(A && W && C && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0, "ri_gemm_rows_bf16: null or unaligned pointer");
    RI_REQUIRE(nt == 1 || nt == 2, "ri_gemm_rows_bf16: nt=%d not 1 or 2", nt);
    RI_REQUIRE(parts >= 1 && parts <= 64, "ri_gemm_rows_bf16: parts=%d not in [1, 64]", parts);
    RI_REQUIRE(parts == 1 || (out_dtype == RI_F32 && !swiglu && part_stride >= (long long)M * ldc),
               "ri_gemm_rows_bf16: partial sums need a float32 stack and no activation");
    const bf16_t* a = (const bf16_t*)A;
    const bf16_t* w = (const bf16_t*)W;
    const size_t ps = parts > 1 ? (size_t)part_stride : 0;
    int rc = 0;
    if (swiglu) {
        RI_REQUIRE(out_dtype == RI_BF16, "ri_gemm_rows_bf16: the fused SwiGLU form writes bfloat16");
        RI_REQUIRE(nt == 1, "ri_gemm_rows_bf16: the SwiGLU form takes one gate and one up tile a wave");
        rc = dispatch_rows<1, true, bf16_t>(a, lda, w, (bf16_t*)C, ldc, M, N, K, 1, 0, groups, stream);
    } else if (out_dtype == RI_BF16) {
        if (nt == 2) rc = dispatch_rows<2, false, bf16_t>(a, lda, w, (bf16_t*)C, ldc, M, N, K, 1, 0, groups, stream);
        else rc = dispatch_rows<1, false, bf16_t>(a, lda, w, (bf16_t*)C, ldc, M, N, K, 1, 0, groups, stream);
    } else if (out_dtype == RI_F32) {
        if (nt == 2) rc = dispatch_rows<2, false, float>(a, lda, w, (float*)C, ldc, M, N, K, parts, ps, groups, stream);
        else rc = dispatch_rows<1, false, float>(a, lda, w, (float*)C, ldc, M, N, K, parts, ps, groups, stream);
    } else {
        return ri_fail("ri_gemm_rows_bf16: unknown output dtype %d", out_dtype);
    }
    if (rc) return rc;
    RI_LAUNCHED("ri_gemm_rows_bf16");
    return 0;
}

// The q/k/v projection of 9..64 tokens with rotation and cache write in the epilogue, as
// ri_gemm_qkv_rope (gemm.hip) does it for fewer rows: W is the same row-permuted weight in tile
// order, C [M, ldc] receives rotated q in its first H * hd columns.  The caller chooses between this and the few-row
// kernel (ops.py, QKV_ROPE_LDS_*, with the figures of both).
//
// Blocks of 32 columns (four pairs of waves) where all of them run at once, one a compute unit; else blocks of 64
// columns (two groups of four waves), half as many: 288 blocks of 32 columns (9216 x 4096) took 27.1 us with 32 rows, 144 of 64 23.0 with 33.
extern "C" int ri_gemm_rows_qkv_rope(const void* A, int lda, const void* W, void* C, int ldc, int M, int K,
                                     int H, int Hkv, int hd, const float* cos_t, const float* sin_t, int table_rows,
                                     const int* positions, const int* row_of_token, void* kc, void* vc,
                                     int num_pages, const int* table, int max_blocks, int page, hipStream_t stream) {
    const int N = (H + 2 * Hkv) * hd;
    RI_REQUIRE(M >= 9 && M <= 64, "ri_gemm_rows_qkv_rope: M=%d not in [9, 64]", M);
    RI_REQUIRE(H > 0 && Hkv > 0 && hd > 0 && hd % 16 == 0 && K > 0 && K % 32 == 0, "ri_gemm_rows_qkv_rope: needs head size %% 16 == 0 and K %% 32 == 0 (hd=%d K=%d)", hd, K);
    RI_REQUIRE(lda >= K && lda % 8 == 0 && ldc >= H * hd, "ri_gemm_rows_qkv_rope: bad leading dimensions");
    RI_REQUIRE(page > 0 && max_blocks > 0 && num_pages > 0 && table_rows > 0, "ri_gemm_rows_qkv_rope: bad cache sizes");
    RI_REQUIRE(A && W && C && cos_t && sin_t && positions && row_of_token && kc && vc && table, "ri_gemm_rows_qkv_rope: null pointer");
    RI_REQUIRE((uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0 && (uintptr_t)cos_t % 16 == 0 && (uintptr_t)sin_t % 16 == 0,
               "ri_gemm_rows_qkv_rope: operands and tables must be 16-byte aligned");
    const RowsRope rp{cos_t, sin_t, positions, row_of_token, table, max_blocks, (bf16_t*)kc, (bf16_t*)vc, H, Hkv, hd, page};
    const bf16_t* a = (const bf16_t*)A;
    const bf16_t* w = (const bf16_t*)W;
    const int groups = (N / 16 + 1) / 2 <= 256 ? 4 : 2;
    int rc;
    if (M <= 16) rc = launch_rows_rope_groups<1>(a, lda, w, (bf16_t*)C, ldc, M, N, K, groups, rp, stream);
    else if (M <= 32) rc = launch_rows_rope_groups<2>(a, lda, w, (bf16_t*)C, ldc, M, N, K, groups, rp, stream);
    else if (M <= 48) rc = launch_rows_rope_groups<3>(a, lda, w, (bf16_t*)C, ldc, M, N, K, groups, rp, stream);
    else rc = launch_rows_rope_groups<4>(a, lda, w, (bf16_t*)C, ldc, M, N, K, groups, rp, stream);
    if (rc) return rc;
    RI_LAUNCHED("ri_gemm_rows_qkv_rope");
    return 0;
}
