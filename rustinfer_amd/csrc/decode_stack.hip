// One decoding step of a whole Llama stack in one launch: up to eight tokens, each the newest of its row.
//
// What bounds it: the weights, read once (1B: 2.5 GB, 360 us at the 6.9 TB/s a kernel that only reads reaches).  As kernels of their own the six
// pieces of a layer (q/k/v with rotation, attention, its merge, o, gate/up, down) take 715 us: each spends 3 to 4 us on the way from the last block
// of the one before to a full stream of its own, 20 us a layer of which the weights take 18.  Here a block a compute unit stays for the whole step
// and reads ahead: weights do not depend on what is computed, so through the end of one product and while the blocks wait for each other's results
// the next product's weights keep coming into LDS until the rings are full (128 KB a unit, 32 MB in all).
// A step then takes, at 100 cached tokens and (2000) and [16000] ones, parts against this launch, us:
//     1B 1 row  721 -> 581 (731 -> 642) [838 -> 730]       3B 1 row  901 -> 795 (899 -> 851) [1095 -> 974]      8B 1 row 1267 -> 1147 (1245 -> 1192) [1410 -> 1297]
//     1B 8 rows 804 -> 669 (878 -> 793) [1502 -> 1345]     3B 8 rows 967 -> 893 (1110 -> 1050) [1999 -> 2013]   8B 8 rows 1323 -> 1234 (1446 -> 1381) [2214 -> 2203]
// What is left above the weights are the five waits of a layer, 2.1 us each from the last block's result to the first block's go on.
//
// Waves of a block: eight multiply (readers), two fill their rings, one is the control wave: it waits for the other blocks, finishes the readers'
// sums and signals.  Loads of a compute unit come back in order, so whatever else the block asks for stands behind the weights under way.  32 KB
// of them under way a unit (two loaders, four rings each, two batches of 2 KB) is the best: 16 to 24 KB 664 to 722 us a step of 1B (too little to
// keep the memory busy), 48 KB 608, 64 KB 610, every wave for itself with all its ring under way 630.
//
// Phases: the embedded rows; a layer's q/k/v, attention, o, gate/up, down; the head.  A phase begins when all items of the phase before it are
// done (where a row's keys are divided, the block that leaves the last part merges them).  What a phase leaves for the next goes through memory:
// stores of agent scope (written through the XCD's L2), acknowledged, then one of eight counters; readers poll the counters and read with plain
// loads, which is sound because every buffer is written once a launch and nobody reads a line of it before it is complete (an L2 of another XCD
// cannot hold an older copy: a launch begins with its L2 clean).  What is read before a phase has ended, the parts of a divided row, lies in lines that
// no other pair of row and key/value head has anything in.  No fence is needed, which would cost tens of microseconds.  The counters lie in
// uncached memory and are polled by scalar loads, which do not stand behind the weights (of cached memory, by vector loads: 650 us).
//
// Which blocks take part is settled at the start: all of the grid, if all are on the chip (the usual case), else those that had arrived
// when the first of them had waited `close_ticks` times what the step takes longer without the rest (of 256 blocks 64: four times); later ones leave at once.
// (Four rows at the 1B sizes beside a kernel of another stream that holds so many units for 1 ms, us, after `close_ticks` whoever is there / this: 128 units 1115 / 1324,
// 200 1865 / 1714, 250 12670 / 1617; 254 for 8 ms 36900 / 8700.)  A step has the whole chip or waits for it: part by part those take 825 us, and of two engines that
// step on two streams, four rows at 1B and eight at 3B, both steps take 1,385 us where launches one after the other take 1,570.  Items are dealt round to those that take part, so every
// block that is waited for is running, whatever else runs on the device, and the products do not depend on their number.  Every wait is bounded
// all the same (the one at the start by `join_ticks`, as one block cannot go on alone; `limit_ticks`, MOST_SPINS): then the launch ends, its logits are NaN, and a word
// in host memory says so.
//
// Products: weights in tile order ([N/16][K/32][64 lanes][8], gemm.hip); K is divided between the eight readers.  Activations (eight rows) are held
// in registers for a phase, two steps of K an operand: columns 0 to 7 of the matrix instruction are the rows at the even step, 8 to 15 at the odd
// one.  o and down take eight columns of weights for two steps a kilobyte, so one instruction makes the sums of both in two quarters of its
// result; q/k/v and the head take 16 columns of one step (two results, half of each used), gate/up eight columns of the gate and the same
// eight of the up half.  (Items of eight columns read 128 of every 256 bytes; with whole tiles wherever there are enough of them a step took 640
// us: fewer items are dealt less evenly.)  The norms are the products' own, as in gemm.hip (RESID, SCALE).
#include "common.h"
#include <math.h>
#include <stdio.h>
#include <mutex>

typedef __bf16 sbf16x8_t __attribute__((ext_vector_type(8)));
typedef float sf32x4_t __attribute__((ext_vector_type(4)));

namespace {

constexpr int WAVES = 8, RING = 16, GROUP = 4;          // waves that multiply; kilobytes of one's ring; kilobytes read from it at a time
constexpr int LOADERS = 2, SERVED = WAVES / LOADERS;    // waves that fill the rings, and rings of each
constexpr int BATCH = 2;                                // kilobytes of a ring asked for at a time; two such under way
constexpr int CONTROL = WAVES, FIRST_LOADER = WAVES + 1, THREADS = (WAVES + 1 + LOADERS) * 64;
constexpr int MAX_ROWS = 8;
constexpr int ATT_VALUES = 512;                         // outputs of a key/value head's queries: (H / Hkv) * head size
constexpr int X_ITEMS = 24;                             // items of eight columns whose residual stream a block can hold
// LDS, in bytes
constexpr int L_RING = 0, L_RED = WAVES * RING * 1024, L_ATT = L_RED + 2 * WAVES * 128 * 4, L_ML = L_ATT + WAVES * ATT_VALUES * 4,
              L_MISC = L_ML + WAVES * 16 * 2 * 4, L_X = L_MISC + 256, L_BYTES = L_X + X_ITEMS * 256;
static_assert(L_BYTES <= 160 * 1024, "a compute unit's LDS");
// words of L_MISC
enum { W_RANK = 0, W_N = 1, W_STOP = 2, W_GO = 3, W_LENGTH = 4, W_ROW = 12, W_LANDED = 20, W_READ = 24, W_SUMS = 32, W_FINISHED = 34, W_MEET = 35,
       W_FIRST = 40 };        // W_FIRST + m: parts of the rows before row m

// control words, a line of 128 bytes each, and behind them counters of the parts of a row's keys; all zero between launches
enum { C_ARRIVED = 0, C_FULL = 8, C_CLOSING = 9, C_STATE = 10, C_MEMBERS = 11, C_DONE = 12, C_LEFT = 20, C_ALL_LEFT = 28, C_PAIRS = 29 };
constexpr int MOST_PAIRS = 256, PAIR_WORDS = 8, CONTROL_WORDS = C_PAIRS * 32 + MOST_PAIRS * PAIR_WORDS;
constexpr unsigned CLOSED = 0x80000000u;
constexpr int MOST_SPINS = 1 << 27;                      // of a word of LDS: some seconds

enum { QKV = 0, O = 1, GATE_UP = 2, DOWN = 3, HEAD = 4, ATTEND = 5, EMBED = 6 };

// The model's table on the device, eight bytes an entry: the weights in the order in which they are read (4 L + 1, the last the
// head's), the norms' weights (2 L + 1: a layer's two, the final one), the norms' eps (2 L + 1, as 64-bit floats).

// A kind of product: its items; kilobytes of an item a wave reads, bytes from one of them to the next and of a tile of 16 columns; added for lanes of
// the second eight columns; whether an item is a whole tile.
struct Kind { int items, units, stride; unsigned tile, second; int whole; };

// offsets within a layer's stretch of scratch, multiples of 256 bytes
struct Offsets { size_t a, ssq, q, at, a2, ssq2, h, po, pml, all; };
__host__ __device__ inline size_t up256(size_t n) { return (n + 255) & ~(size_t)255; }
// A part of a row's keys, for the G queries of a key/value head, leaves its unnormalised outputs (G x hd floats) in a slot of `po` and their maxima and sums in one of
// `pml`.  A row is merged when its own parts are there, while others still write theirs: a slot of either is whole lines of its own (128 bytes), or a merge
// would bring a line into its L2 in which another row's entries are not yet what a merge on the same XCD then reads.
constexpr size_t LINE = 128;
__host__ __device__ inline size_t slot_outputs(int G, int hd) { return (size_t)G * hd * 4; }                             // bytes; hd is 64 or 128
constexpr size_t SLOT_SUMS = LINE;                                                                                       // G pairs of floats, G <= 16
static_assert(64 * 4 % LINE == 0 && 16 * 8 <= SLOT_SUMS, "a slot is whole lines");
// A row's keys are divided between blocks in parts of `share` keys or fewer, PART_KEYS at least: the waves of all of a row's parts take spans of SPAN keys in turn.
constexpr int SPAN = 32, PART_KEYS = WAVES * SPAN, WHOLE_KEYS = 2 * PART_KEYS;
__host__ __device__ inline int parts_of(int len, int share) { return len <= share ? 1 : (len + share - 1) / share; }
__host__ __device__ inline Offsets stack_offsets(int M, int d, int ff, int H, int Hkv, int hd, int blocks) {
    Offsets o;
    size_t at = 0;
    auto take = [&](size_t n) { const size_t r = at; at += up256(n); return r; };
    o.a = take((size_t)M * d * 2); o.ssq = take((size_t)M * (d / 8) * 4);
    o.q = take((size_t)M * H * hd * 2); o.at = take((size_t)M * H * hd * 2);
    o.a2 = take((size_t)M * d * 2); o.ssq2 = take((size_t)M * (d / 8) * 4);
    o.h = take((size_t)M * ff * 2);
    o.po = take(blocks * slot_outputs(H / Hkv, hd)); o.pml = take(blocks * SLOT_SUMS);                       // (where rows are divided, a block has one part)
    o.all = at;
    return o;
}

struct StackArgs {
    const uint64_t* model;
    int L, M, d, ff, H, Hkv, V, n_f32;
    const int* ids; const int* device_tokens; const bf16_t* table;                        // embedding
    const int* positions; const int* row_of_token; const int* kv_lens; const int* blocks; int max_blocks;
    const float* cos_t; const float* sin_t;
    bf16_t* kc; bf16_t* vc; size_t k_layer, v_layer;    // caches of the first layer, and values from one layer's to the next's
    float scale;
    float* logits; int ld_logits;
    char* scratch; size_t layer_bytes;                  // buffers that the phases leave for each other, a stretch a layer
    float* x;                                           // [d / 8][8][8] the residual stream, by items
    unsigned* control; int expect;                      // blocks that may take part: a multiple of 8
    unsigned* gave_up;                                  // host memory: set by a launch that did not run to its end
    unsigned long long close_ticks, join_ticks, limit_ticks;
    Offsets off;
    Kind kinds[5];
};
// The launch's arguments, read where they are used by scalar loads: kept in registers, all of them at once are too many.
typedef const __attribute__((address_space(4))) StackArgs* Args;
__device__ __forceinline__ Args again(Args p) {
    uint64_t v = (uint64_t)p;
    asm volatile("" : "+s"(v));
    return (Args)v;
}

__device__ __forceinline__ unsigned ld_agent(const unsigned* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <typename T> __device__ __forceinline__ void st_agent(T* p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ unsigned add_agent(unsigned* p, unsigned v) { return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// The block's waves wait for each other through words of LDS that only grow: a barrier would have to be passed by those that fill the rings too.
// Reads and writes of them are written out: around ordinary ones the compiler waits for all loads on their way into LDS.
__device__ __forceinline__ unsigned lds_address(const void* p) { return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) void*)p; }
__device__ __forceinline__ int word_at(unsigned at) {                     // the same for all lanes
    int v;
    asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"(at) : "memory");
    return __builtin_amdgcn_readfirstlane(v);
}
// what the wave has put into LDS before is there when the word says so
__device__ __forceinline__ void set_word(unsigned at, int v) { asm volatile("s_waitcnt lgkmcnt(0)\n\tds_write_b32 %0, %1" :: "v"(at), "v"(v) : "memory"); }
__device__ __forceinline__ void add_word(unsigned at, int lane) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (lane == 0) asm volatile("ds_add_u32 %0, %1" :: "v"(at), "v"(1) : "memory");
}
// Until the word is at least `least`, or the block is to stop: after some seconds of waiting it is.
__device__ __forceinline__ void wait_word(unsigned misc, int word, int least) {
    int v, stop, left = MOST_SPINS;
    do {
        asm volatile("ds_read_b32 %0, %2\n\tds_read_b32 %1, %3\n\ts_waitcnt lgkmcnt(0)" : "=&v"(v), "=&v"(stop) : "v"(misc + word * 4), "v"(misc + W_STOP * 4) : "memory");
    } while (__builtin_amdgcn_readfirstlane(v) < least && __builtin_amdgcn_readfirstlane(stop) == 0 && --left > 0);
    if (left == 0) set_word(misc + W_STOP * 4, 1);
}
// a wave's own stores are where everyone sees them
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// The model's table is read by scalar loads: it does not change, and a wave's counter of vector loads is the ring's.
typedef const __attribute__((address_space(4))) uint64_t* ModelPtr;
__device__ __forceinline__ const void* weight_at(Args A, int p) { return reinterpret_cast<const void*>(((ModelPtr)(uintptr_t)A->model)[p]); }
__device__ __forceinline__ const void* norm_at(Args A, int i) { return reinterpret_cast<const void*>(((ModelPtr)(uintptr_t)A->model)[4 * A->L + 1 + i]); }
__device__ __forceinline__ float eps_at(Args A, int i) {
    return (float)__builtin_bit_cast(double, (uint64_t)((ModelPtr)(uintptr_t)A->model)[6 * A->L + 2 + i]);
}

// (registers that hold something from here on, whatever it is: not from the phase before)
template <typename T, int N> __device__ __forceinline__ void begin_registers(T (&a)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "=v"(a[i]));
}
// (the same number, not known to be: what follows from it is made where it is needed and not kept in registers across the phases)
__device__ __forceinline__ int hidden(int v) {
    v = __builtin_amdgcn_readfirstlane(v);
    asm volatile("" : "+s"(v));
    return v;
}
__device__ __forceinline__ int hidden_lane(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// What fills the rings of SERVED waves: the weights of all their items of all phases, one after the other, as fast as the rings are read, two
// batches of each under way.
struct Loader {
    const Args K;
    const int rank, n, first, lane;                     // first: of the waves it serves
    char* rings;
    const unsigned misc;
    // where the next kilobyte of the first ring lies; all but lane_off are the same in all lanes
    const char* at = nullptr;
    const char* item_at = nullptr;
    unsigned lane_off = 0, step = 0, wave_step = 0;
    int left = 0, units = 0, stride = 0, item = 0, items = 0, phase = -1;      // phase: of the products' 4 L + 1
    bool ended = false;

    __device__ __forceinline__ Loader(Args K_, int rank_, int n_, int first_, int lane_, char* rings_, unsigned misc_)
        : K(K_), rank(rank_), n(n_), first(first_), lane(lane_), rings(rings_), misc(misc_) { next_item(); }

    __device__ __forceinline__ void next_item() {
        item += n;
        item_at += step;
        if (item >= items) {
            const Args A = again(K);
            const int last = 4 * A->L;
#pragma unroll 1
            do {
                if (++phase > last) { ended = true; return; }
                items = A->kinds[phase == last ? HEAD : phase & 3].items;
            } while (rank >= items);
            const auto* k = &A->kinds[phase == last ? HEAD : phase & 3];
            item = rank;
            units = k->units;
            stride = k->stride;
            const unsigned tile = k->tile;
            const int shift = k->whole ? 0 : 1;           // (half tiles: a block keeps its half from one to the next, as n is even)
            step = (unsigned)(n >> shift) * tile;
            wave_step = tile / WAVES;
            item_at = reinterpret_cast<const char*>(weight_at(A, phase)) + (unsigned)(rank >> shift) * tile + wave_step * (unsigned)first;
            lane_off = (unsigned)((lane >> 4) * 256 + (lane & 7) * 16) + (shift ? (unsigned)(rank & 1) * 128u : 0u) + ((lane & 8) ? k->second : 0u);
        }
        at = item_at;
        left = units;
    }
    // at most LEAVE kilobytes of each ring under way
    template <int LEAVE> __device__ __forceinline__ void leave() { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(LEAVE * SERVED) : "memory"); }
    __device__ __forceinline__ void run() {
        int row = 0, landed = 0, read = 0;                // kilobytes of a ring asked for, there, and read by all
        for (;;) {
            if (!ended && row - read <= RING - BATCH && row - landed <= BATCH) {
#pragma unroll 1
                for (int u = 0; u < BATCH && !ended; ++u) {
                    char* to = rings + (first * RING + (row & (RING - 1))) * 1024;
#pragma unroll
                    for (int r = 0; r < SERVED; ++r)
                        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(at + wave_step * r + lane_off),
                                                         (__attribute__((address_space(3))) void*)(to + r * RING * 1024), 16, 0, 2);
                    ++row;
                    at += stride;
                    if (--left == 0) next_item();
                }
                continue;
            }
            if (landed < row) {
                landed = row - landed > BATCH ? row - BATCH : row;
                if (landed < row) leave<BATCH>();
                else leave<0>();
                set_word(misc + (W_LANDED + first / SERVED) * 4, landed);
            } else {
                if (ended || word_at(misc + W_STOP * 4)) return;
                __builtin_amdgcn_s_sleep(1);
            }
            int v;
            asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"(misc + (W_READ + first + (lane & (SERVED - 1))) * 4) : "memory");
            v = min(v, __builtin_amdgcn_mov_dpp(v, 0xb1, 0xf, 0xf, true));     // lane ^ 1
            v = min(v, __builtin_amdgcn_mov_dpp(v, 0x4e, 0xf, 0xf, true));     // lane ^ 2
            read = __builtin_amdgcn_readfirstlane(v);
        }
    }
};
static_assert(BATCH * SERVED < 64 && SERVED == 4, "the counter of loads, and the smallest of four words above");

// One of the waves that multiply: sums over its share of K.
struct Reader {
    const int rank, n, wave;
    int lane;
    const char* ring;                                   // this wave's, in LDS
    float* red;                                         // [2][WAVES][128]
    const unsigned misc;
    int pos = 0, sums = 0;                              // kilobytes read; items done

    // the next `count` kilobytes (at most GROUP) in registers
    __device__ __forceinline__ void take(sbf16x8_t (&w)[GROUP], int count) {
        wait_word(misc, W_LANDED + wave / SERVED, pos + count);
#pragma unroll
        for (int u = 0; u < GROUP; ++u) w[u] = *reinterpret_cast<const sbf16x8_t*>(ring + ((pos + u) & (RING - 1)) * 1024 + lane * 16);
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]) :: "memory");
        pos += count;
        set_word(misc + (W_READ + wave) * 4, pos);
    }
    // operands of the rows of act [M][K]: of this wave's share of K two steps of 32 an operand, columns 0 to 7 the first
    template <int NF> __device__ __forceinline__ void load_rows(sbf16x8_t (&a)[NF], const bf16_t* act, int F, int M) {
        const int depth = F * (64 * WAVES), c = lane & 15, row = min(c & 7, M - 1);     // (rows beyond the last make columns nobody reads)
        const bf16_t* p = act + (size_t)row * depth + (size_t)wave * F * 64 + (c >> 3) * 32 + (lane >> 4) * 8;
#pragma unroll
        for (int f = 0; f < NF; ++f)
            if (f < F) a[f] = *reinterpret_cast<const sbf16x8_t*>(p + f * 64);
    }
    // A phase's items against rows of K values; the control wave finishes them.
    template <int NF, bool PAIR> __device__ __forceinline__ void product(const bf16_t* act, int count, int all, int M) {
        if (rank >= count) return;
        lane = hidden_lane(lane);
        sbf16x8_t a[NF];
        begin_registers(a);
        load_rows<NF>(a, act, hidden(all), M);
        const int c = lane & 15, g = lane >> 4;
#pragma unroll 1
        for (int i = rank; i < count; i += n) {
            sf32x4_t acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
            sbf16x8_t w[GROUP];
            const int F = hidden(all);
            if constexpr (PAIR) {
#pragma unroll
                for (int f = 0; f < NF; f += GROUP) {
                    if (f >= F) continue;
                    take(w, min(GROUP, F - f));
#pragma unroll
                    for (int u = 0; u < GROUP; ++u)
                        if (f + u < NF && f + u < F) {
                            if (u & 1) acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u], a[f + u < NF ? f + u : 0], acc1, 0, 0, 0);
                            else acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u], a[f + u < NF ? f + u : 0], acc0, 0, 0, 0);
                        }
                }
            } else {
#pragma unroll
                for (int f = 0; f < NF; f += GROUP / 2) {
                    if (f >= F) continue;
                    take(w, 2 * min(GROUP / 2, F - f));
#pragma unroll
                    for (int u = 0; u < GROUP / 2; ++u)
                        if (f + u < NF && f + u < F) {
                            acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[2 * u], a[f + u < NF ? f + u : 0], acc0, 0, 0, 0);
                            acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[2 * u + 1], a[f + u < NF ? f + u : 0], acc1, 0, 0, 0);
                        }
                }
            }
            // element i of lane 16 g + c is column 4 g + i of the weights, column c of the rows' operand: [column][row] of the item
            // (its place is free when the item before the last is finished)
            wait_word(misc, W_FINISHED, sums - 1);
            float* out = red + ((sums & 1) * WAVES + wave) * 128;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (PAIR) {
                    const float s = acc0[e] + acc1[e];
                    const float both = s + __int_as_float(__builtin_amdgcn_ds_bpermute(((lane + 40) & 63) * 4, __float_as_int(s)));
                    if (g < 2 && c < 8) out[(g * 4 + e) * 8 + c] = both;
                } else {
                    const float s = c < 8 ? acc0[e] : acc1[e];
                    const float both = s + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(s), 0x128, 0xf, 0xf, true));     // lane ^ 8
                    if (c < 8) out[(g * 4 + e) * 8 + c] = both;
                }
            }
            added();
        }
    }
    // An item's sums are there.  A counter for every other item: a wave may be one ahead of another, and a count of all items would take its
    // next one for the other's share of this one.
    __device__ __forceinline__ void added() {
        add_word(misc + (W_SUMS + (sums & 1)) * 4, lane);
        ++sums;
    }
    // all the waves that multiply
    int meets = 0;
    __device__ __forceinline__ void meet() {
        add_word(misc + W_MEET * 4, lane);
        meets += WAVES;
        wait_word(misc, W_MEET, meets);
    }
};

// How the rows' keys are divided: between all blocks by the rows' lengths, so that the longest share, which the others wait for, is as short as it can be (with as many parts
// for every row, 8 rows of which one had 16,000 keys and the others 100 took 1,644 us at the 3B sizes, now 1,113, part by part 1,145; 4,000 and 100 1,103 / 1,002 / 1,069).  The share
// goes by spans: by PART_KEYS eight rows of 2,100 keys had three parts each where four fit, 1,402 us a step at the 8B sizes, now 1,387.  Not where the longest row has
// WHOLE_KEYS keys or fewer: a merge costs more than it gives.  `total` of a share: the parts of all rows.
template <typename F> __device__ __forceinline__ int share_of(F total, int longest, int budget, int rows, int lane) {
    if (longest <= WHOLE_KEYS || budget <= rows) return 0x7fffffff;
    for (int from = PART_KEYS, unit = SPAN; unit < 1 << 24; from += 64 * unit, unit *= 2) {        // (the 64 lanes try one each)
        const unsigned long long fits = __ballot(total(from + unit * lane) <= budget);
        if (fits) return from + unit * __builtin_ctzll(fits);
    }
    return 0x7fffffff;
}

// A span's keys and values as the matrix instructions read them: tile e of the keys holds, in row r, key 8 (r / 4) + 4 e + r % 4.
template <int HD> struct SpanOf { sbf16x8_t k[2][HD / 32], v[HD / 16]; };

// One wave's share of one part of a row's keys for the queries of one key/value head, in the order of attn_decode_split_kernel: what it
// leaves are its maximum, its sum and its unnormalised outputs, in LDS.  Loads are under no lane's condition: beyond the row they read its last page
// again, their scores are put to -inf and their values to zero.
template <int HD>
struct Attention {
    const bf16_t *kc, *vc;                              // of the key/value head
    const __attribute__((address_space(4))) int* pages; // of the row
    size_t page_step;                                   // values from one page to the next
    int len, lane;
    SpanOf<HD> s;

    __device__ __forceinline__ void keys(int sp) {
        const int col = lane & 15, grp = lane >> 4, last = len - 1, k0 = sp * SPAN;
        const int p0 = pages[k0 >> 4], p1 = pages[min(k0 + 16, last) >> 4];
        const bf16_t* kt = kc + (size_t)(col < 8 ? p0 : p1) * page_step + (((col >> 2) * 8 + (col & 3)) & 15) * HD + grp * 8;
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int kk = 0; kk < HD / 32; ++kk) s.k[e][kk] = ld_stream16<sbf16x8_t>(kt + e * 4 * HD + kk * 32);
    }
    __device__ __forceinline__ void values(int sp) {
        const int col = lane & 15, grp = lane >> 4, last = len - 1, k0 = sp * SPAN;
        const int p0 = pages[k0 >> 4], p1 = pages[min(k0 + 16, last) >> 4];
        const bf16_t* vt = vc + (size_t)(grp < 2 ? p0 : p1) * page_step + col * 16 + (grp & 1) * 8;
#pragma unroll
        for (int db = 0; db < HD / 16; ++db) s.v[db] = ld_stream16<sbf16x8_t>(vt + db * 256);
    }
    // q: of the group's G heads; asked: the first span's keys and values have been asked for
    __device__ __forceinline__ void run(const bf16_t* q, int G, float scale, int first, int step, bool asked, float* so, float* ml) {
        const int col = lane & 15, grp = lane >> 4;
        const int spans = (len + SPAN - 1) / SPAN;
        const sbf16x8_t zero = {};
        if (first < spans && !asked) { keys(first); values(first); }
        sbf16x8_t qf[HD / 32];
#pragma unroll
        for (int kk = 0; kk < HD / 32; ++kk) {
            qf[kk] = *reinterpret_cast<const sbf16x8_t*>(q + min(col, G - 1) * HD + kk * 32 + grp * 8);
            if (col >= G) qf[kk] = zero;
        }
        sf32x4_t o[HD / 16];
#pragma unroll
        for (int db = 0; db < HD / 16; ++db) o[db] = sf32x4_t{0.f, 0.f, 0.f, 0.f};
        float m_run = -INFINITY, l_run = 0.f;
#pragma unroll 1
        for (int sp = first; sp < spans; sp += step) {
            const int k0 = sp * SPAN;
            sf32x4_t st[2];
            float top = m_run;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                st[e] = sf32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kk = 0; kk < HD / 32; ++kk) st[e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(s.k[e][kk], qf[kk], st[e], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    st[e][i] = k0 + grp * 8 + e * 4 + i < len ? st[e][i] * scale : -INFINITY;
                    top = fmaxf(top, st[e][i]);
                }
            }
            if (sp + step < spans) keys(sp + step);
            else { begin_registers(s.k[0]); begin_registers(s.k[1]); }
            top = fmaxf(top, __shfl_xor(top, 16, 64));
            top = fmaxf(top, __shfl_xor(top, 32, 64));
            const float base = top == -INFINITY ? 0.f : top;  // (scores that are all -inf weigh nothing)
            float sum = 0.f;
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
                for (int i = 0; i < 4; ++i) { st[e][i] = __expf(st[e][i] - base); sum += st[e][i]; }
            sum += __shfl_xor(sum, 16, 64);
            sum += __shfl_xor(sum, 32, 64);
            const float alpha = __expf(m_run - base);
            l_run = l_run * alpha + sum;
            m_run = top;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float ai = __shfl(alpha, grp * 4 + i, 64);
#pragma unroll
                for (int db = 0; db < HD / 16; ++db) o[db][i] *= ai;
            }
            sbf16x8_t hi, lo;                             // the weights as the sum of two bfloat16
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float p = st[i >> 2][i & 3];
                hi[i] = (__bf16)p;
                lo[i] = (__bf16)(p - (float)hi[i]);
            }
            if (k0 + SPAN > len) {                        // positions never written may hold anything, NaN included
                const int n = len - k0 - grp * 8;
                ri_u32x4_t keep;
#pragma unroll
                for (int w = 0; w < 4; ++w) keep[w] = (2 * w < n ? 0xffffu : 0u) | (2 * w + 1 < n ? 0xffff0000u : 0u);
#pragma unroll
                for (int db = 0; db < HD / 16; ++db) s.v[db] = __builtin_bit_cast(sbf16x8_t, __builtin_bit_cast(ri_u32x4_t, s.v[db]) & keep);
            }
#pragma unroll
            for (int db = 0; db < HD / 16; ++db) {
                o[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, s.v[db], o[db], 0, 0, 0);
                o[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, s.v[db], o[db], 0, 0, 0);
            }
            if (sp + step < spans) values(sp + step);
            else begin_registers(s.v);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int qi = grp * 4 + i;
            if (qi < G) {
#pragma unroll
                for (int db = 0; db < HD / 16; ++db) so[qi * HD + db * 16 + col] = o[db][i];
            }
        }
        if (grp == 0) { ml[col] = m_run; ml[16 + col] = l_run; }
    }
};

// The control wave's wait for everything up to `target` arrivals.
__device__ __forceinline__ bool all_done(Args A, unsigned target, int lane, unsigned long long begun) {
    if (A->limit_ticks == 0) return false;               // (no waiting at all)
    for (unsigned spin = 1;; ++spin) {
        unsigned c0, c1, c2, c3, c4, c5, c6, c7;
        asm volatile("s_load_dword %0, %8, 0x0 glc\n\ts_load_dword %1, %8, 0x80 glc\n\ts_load_dword %2, %8, 0x100 glc\n\ts_load_dword %3, %8, 0x180 glc\n\t"
                     "s_load_dword %4, %8, 0x200 glc\n\ts_load_dword %5, %8, 0x280 glc\n\ts_load_dword %6, %8, 0x300 glc\n\ts_load_dword %7, %8, 0x380 glc\n\t"
                     "s_waitcnt lgkmcnt(0)"
                     : "=&s"(c0), "=&s"(c1), "=&s"(c2), "=&s"(c3), "=&s"(c4), "=&s"(c5), "=&s"(c6), "=&s"(c7) : "s"(A->control + C_DONE * 32) : "memory");
        if (c0 + c1 + c2 + c3 + c4 + c5 + c6 + c7 >= target) return true;
        if ((spin & 255) == 0 && __builtin_amdgcn_readfirstlane(wall_clock64() - begun > A->limit_ticks ? 1 : 0)) return false;
    }
}

__device__ __forceinline__ float norm_weight(Args A, const void* w, int i) {
    return A->n_f32 ? reinterpret_cast<const float*>(w)[i] : bf16_to_f32(reinterpret_cast<const bf16_t*>(w)[i]);
}

// of the eight lanes of a row: the neighbour's value, and all of them added up
__device__ __forceinline__ float neighbour(float v) { return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xb1, 0xf, 0xf, true)); }
__device__ __forceinline__ float sum_of_eight(float v) {
    v += neighbour(v);
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4e, 0xf, 0xf, true));
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xf, 0xf, true));
    return v;
}

// The parts of a row's keys for the G queries of a key/value head, by one wave: eight values a lane.  What is asked for stands behind the weights under way, so it
// is asked for at once: maxima, sums and outputs of eight parts, those of head size 64 by two halves of the wave where 32 lanes hold a part (and by four
// parts a turn, as that kernel gets slower with the registers of eight: 580 -> 615 us a step of one row).  us a step of one row of 8,000 keys, a trip for the maxima
// and one for every four parts / this: 1B 707 / 689, 3B 993 / 908, 8B 1311 / 1242.
template <int HD>
__device__ __forceinline__ void merge(const char* po, const char* pml, size_t first, int step, int parts, int G, bf16_t* out, int lane) {
    constexpr int TURN = HD == 64 ? 4 : 8;
    const bool halves = HD == 64 && G * HD <= 256;
    const int e = (halves ? lane & 31 : lane) * 8, qi = e / HD, by = halves ? 2 : 1;
    if (e >= G * HD) return;
    const char* ml = pml + first * SLOT_SUMS + qi * 8;
    const char* o = po + first * slot_outputs(G, HD) + (size_t)e * 4;
    const size_t ml_step = step * SLOT_SUMS, o_step = step * slot_outputs(G, HD);
    float top = -INFINITY, sum = 0.f, v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int p0 = halves ? lane >> 5 : 0; p0 < parts; p0 += TURN * by) {
        float2 two[TURN];
        float4 a[TURN], b[TURN];
#pragma unroll
        for (int u = 0; u < TURN; ++u) {
            const size_t p = min(p0 + u * by, parts - 1);                  // (beyond the last: again, and without weight)
            two[u] = *reinterpret_cast<const float2*>(ml + p * ml_step);
            a[u] = *reinterpret_cast<const float4*>(o + p * o_step);
            b[u] = *reinterpret_cast<const float4*>(o + p * o_step + 16);
        }
        __builtin_amdgcn_sched_barrier(0);                                 // (all of them under way before the first is waited for)
        float most = top;
#pragma unroll
        for (int u = 0; u < TURN; ++u) most = fmaxf(most, two[u].x);
        const float base = most == -INFINITY ? 0.f : most, alpha = __expf(top - base);
        top = most;
        sum *= alpha;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] *= alpha;
#pragma unroll
        for (int u = 0; u < TURN; ++u) {
            const bool there = p0 + u * by < parts;
            const float w = !there || two[u].x == -INFINITY ? 0.f : __expf(two[u].x - base);
            sum += w * two[u].y;
            if (!there) a[u] = b[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            v[0] += w * a[u].x; v[1] += w * a[u].y; v[2] += w * a[u].z; v[3] += w * a[u].w;
            v[4] += w * b[u].x; v[5] += w * b[u].y; v[6] += w * b[u].z; v[7] += w * b[u].w;
        }
    }
    if (halves) {
        const float other = __shfl_xor(top, 32, 64), most = fmaxf(top, other), base = most == -INFINITY ? 0.f : most;
        const float mine = __expf(top - base), theirs = __expf(other - base);
        sum = sum * mine + __shfl_xor(sum, 32, 64) * theirs;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = v[i] * mine + __shfl_xor(v[i], 32, 64) * theirs;
        if (lane >= 32) return;
    }
#pragma unroll
    for (int i = 0; i < 8; i += 2)
        st_agent(reinterpret_cast<unsigned*>(out + e + i), (unsigned)f32_to_bf16(v[i] / sum) | ((unsigned)f32_to_bf16(v[i + 1] / sum) << 16));
}

// two neighbouring columns' values, bfloat16, by the lane of the even one
__device__ __forceinline__ void store_pair(bf16_t* p, float v, bool live, int lane) {
    const float other = neighbour(v);
    if (live && !(lane & 1)) st_agent(reinterpret_cast<unsigned*>(p), (unsigned)f32_to_bf16(v) | ((unsigned)f32_to_bf16(other) << 16));
}

template <int HD, int NF_D, int NF_FF>
__global__ __launch_bounds__(THREADS) void decode_stack_kernel(const StackArgs) {
    const Args A = (Args)__builtin_amdgcn_kernarg_segment_ptr();
    extern __shared__ __align__(16) char lds[];
    float* red = reinterpret_cast<float*>(lds + L_RED);
    float* att_o = reinterpret_cast<float*>(lds + L_ATT);
    float* att_ml = reinterpret_cast<float*>(lds + L_ML);
    volatile int* misc = reinterpret_cast<volatile int*>(lds + L_MISC);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int shard = blockIdx.x & 7;
    unsigned long long begun = wall_clock64();
    bool given_up = false;                                // of the control wave
    unsigned* ctl = again(A)->control;
    if (wave == CONTROL) {
        misc[lane] = 0;
        if (lane < MAX_ROWS) {
            const int b = lane < again(A)->M ? again(A)->row_of_token[lane] : -1;
            misc[W_LENGTH + lane] = b >= 0 ? max(0, min(again(A)->kv_lens[b], again(A)->positions[lane] + 1)) : 0;
            misc[W_ROW + lane] = b;
        }
        // who takes part
        const unsigned per = (unsigned)again(A)->expect / 8;
        unsigned got = 0;
        if (lane == 0) got = add_agent(ctl + (C_ARRIVED + shard) * 32, 1u);
        got = (unsigned)__builtin_amdgcn_readfirstlane((int)got);
        int rank = 0, n = 0;
        if (!(got & CLOSED)) {
            if (got == per - 1 && lane == 0) add_agent(ctl + C_FULL * 32, 1u);
            bool tried = false;
            for (;;) {
                const unsigned v = lane < 2 ? ld_agent(ctl + (lane == 0 ? C_FULL : C_STATE) * 32) : 0u;
                const unsigned full = (unsigned)__builtin_amdgcn_readlane((int)v, 0), state = (unsigned)__builtin_amdgcn_readlane((int)v, 1);
                if (full == 8) { rank = (int)(shard * per + got); n = again(A)->expect; break; }
                if (state != 0) {
                    const unsigned w = lane < 9 ? ld_agent(ctl + C_MEMBERS * 32 + lane) : 0u;
                    n = __builtin_amdgcn_readlane((int)w, 8);
                    rank = __shfl((int)w, shard, 64) + (int)got;
                    rank = __builtin_amdgcn_readfirstlane(rank);
                    break;
                }
                // (two blocks are the least that can go on: until then others hold the chip)
                const unsigned long long waited = wall_clock64() - begun;
                if (__builtin_amdgcn_readfirstlane(waited > again(A)->join_ticks ? 1 : 0)) { given_up = true; break; }
                if (!tried && __builtin_amdgcn_readfirstlane(waited > again(A)->close_ticks ? 1 : 0)) {
                    unsigned here = 0;
                    if (lane < 8) here = ld_agent(ctl + (C_ARRIVED + lane) * 32) & ~CLOSED;
                    unsigned sum = 0;
                    for (int i = 0; i < 8; ++i) sum += (unsigned)__builtin_amdgcn_readlane((int)here, i);
                    if (sum < 2 || __builtin_amdgcn_readfirstlane(waited * sum < again(A)->close_ticks * (unsigned)again(A)->expect ? 1 : 0)) continue;
                    tried = true;
                    unsigned first = 0;
                    if (lane == 0) first = add_agent(ctl + C_CLOSING * 32, 1u);
                    if (__builtin_amdgcn_readfirstlane((int)first) == 0) {
                        unsigned c = 0;
                        if (lane < 8) c = __hip_atomic_fetch_or(ctl + (C_ARRIVED + lane) * 32, CLOSED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        unsigned before = 0, sum = 0;
                        for (int i = 0; i < 8; ++i) {
                            const unsigned ci = (unsigned)__builtin_amdgcn_readlane((int)c, i);
                            if (i < lane) before += ci;
                            sum += ci;
                        }
                        if (lane < 9) st_agent(ctl + C_MEMBERS * 32 + lane, lane < 8 ? before : sum & ~1u);
                        stores_done();
                        if (lane == 0) st_agent(ctl + C_STATE * 32, 1u);
                    }
                }
            }
        }
        if (rank >= n) n = 0;                             // (an odd one out: items of half a tile keep their half from one to the next)
        if (lane == 0) { misc[W_RANK] = rank; misc[W_N] = n; }
        if (n > 0) {
            const int M = again(A)->M, len = lane < MAX_ROWS ? misc[W_LENGTH + lane] : 0;
            int longest = 0;
            for (int m = 0; m < M; ++m) longest = max(longest, __builtin_amdgcn_readlane(len, m));
            const int share = share_of([&](int s) {
                int sum = 0;
                for (int m = 0; m < M; ++m) sum += parts_of(__builtin_amdgcn_readlane(len, m), s);
                return sum;
            }, longest, n / again(A)->Hkv, M, lane);
            int first = 0;
            for (int m = 0; m < M; ++m) first += m < lane ? parts_of(__builtin_amdgcn_readlane(len, m), share) : 0;
            if (lane <= MAX_ROWS) misc[W_FIRST + lane] = first;
        }
        begun = wall_clock64();
    }
    __syncthreads();
    const int rank = __builtin_amdgcn_readfirstlane(misc[W_RANK]), n = __builtin_amdgcn_readfirstlane(misc[W_N]);
    const unsigned words = lds_address(lds + L_MISC);
    if (n > 0) {
        const int H = again(A)->H, Hkv = again(A)->Hkv, G = H / Hkv, q_dim = H * HD, M = again(A)->M;
        const int jobs = __builtin_amdgcn_readfirstlane(misc[W_FIRST + M]) * Hkv;                  // parts of rows, by key/value heads
        // the row of a job, of which this is part `part` of `parts`
        auto row_of = [&](int job, int& part, int& parts) {
            const int at = job / Hkv;
            int m = 0, from = 0, to = __builtin_amdgcn_readfirstlane(misc[W_FIRST + 1]);
            while (at >= to) { ++m; from = to; to = __builtin_amdgcn_readfirstlane(misc[W_FIRST + 1 + m]); }
            part = at - from;
            parts = to - from;
            return m;
        };
        if (wave >= FIRST_LOADER) {
            Loader loader(A, rank, n, (wave - FIRST_LOADER) * SERVED, lane, lds + L_RING, words);
            loader.run();
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // nothing may be on its way into LDS when the block ends
        } else if (wave < WAVES) {
            Reader s{rank, n, wave, lane, lds + L_RING + wave * RING * 1024, red, words};
            int kind = QKV, l = 0, begun_phases = 0;
#pragma unroll 1
            for (;;) {
                // the phases in order; what a phase reads is behind its barrier
                const Args P = again(A);
                char* base = P->scratch + (size_t)l * P->layer_bytes;
                bf16_t* attn = reinterpret_cast<bf16_t*>(base + P->off.at);
                char* po = base + P->off.po;
                char* pml = base + P->off.pml;
                if (kind == ATTEND) {
                    // attention of this block's first job: what does not depend on this step is asked for now
                    const int lane = hidden_lane((int)threadIdx.x) & 63;
                    Attention<HD> at;
                    begin_registers(at.s.k[0]);
                    begin_registers(at.s.k[1]);
                    begin_registers(at.s.v);
                    const int rank = hidden(s.rank), n = hidden(s.n);
                    int job = rank, m = 0, g = 0, part = 0, parts = 1;
                    bool asked = false;
                    auto take_job = [&]() {
                        m = row_of(job, part, parts);
                        g = job % Hkv;
                        const int b = __builtin_amdgcn_readfirstlane(misc[W_ROW + m]);
                        at.len = __builtin_amdgcn_readfirstlane(misc[W_LENGTH + m]);
                        at.lane = lane;
                        at.page_step = (size_t)Hkv * (16 * HD);
                        at.kc = P->kc + (size_t)l * P->k_layer + (size_t)g * (16 * HD);
                        at.vc = P->vc + (size_t)l * P->v_layer + (size_t)g * (16 * HD);
                        at.pages = (const __attribute__((address_space(4))) int*)(uintptr_t)(P->blocks + (size_t)max(b, 0) * P->max_blocks);
                    };
                    if (job < jobs) {
                        take_job();
                        const int sp = part * WAVES + wave;
                        asked = (sp + 1) * SPAN < at.len;      // (not the span that this step's own key is in)
                        if (asked) { at.keys(sp); at.values(sp); }
                    }
                    wait_word(words, W_GO, ++begun_phases);
                    if (word_at(words + W_STOP * 4)) break;
                    const bf16_t* q = reinterpret_cast<const bf16_t*>(base + P->off.q);
                    for (; job < jobs; job += n, asked = false) {
                        if (job != rank) take_job();
                        const bool some = at.len > 0;
                        if (some) at.run(q + (size_t)m * q_dim + (size_t)g * G * HD, G, P->scale, part * WAVES + wave, parts * WAVES, asked, att_o + wave * ATT_VALUES, att_ml + wave * 32);
                        s.meet();
                        const int e = (wave * 64 + lane) * 2;
                        if (e < G * HD) {
                            const int qi = e / HD, dd = e - qi * HD;
                            float v0 = 0.f, v1 = 0.f, top = -INFINITY, sum = 0.f;
                            if (some) {
#pragma unroll
                                for (int w = 0; w < WAVES; ++w) top = fmaxf(top, att_ml[w * 32 + qi]);
#pragma unroll
                                for (int w = 0; w < WAVES; ++w) {
                                    const float mw = att_ml[w * 32 + qi], wt = mw == -INFINITY ? 0.f : __expf(mw - top);
                                    sum += wt * att_ml[w * 32 + 16 + qi];
                                    const float2 ov = *reinterpret_cast<const float2*>(att_o + w * ATT_VALUES + e);
                                    v0 += wt * ov.x;
                                    v1 += wt * ov.y;
                                }
                            }
                            if (parts == 1) {
                                if (some) { v0 /= sum; v1 /= sum; }
                                st_agent(reinterpret_cast<unsigned*>(attn + (size_t)m * q_dim + (size_t)g * G * HD + e),
                                         (unsigned)f32_to_bf16(v0) | ((unsigned)f32_to_bf16(v1) << 16));
                            } else {
                                st_agent(reinterpret_cast<unsigned long long*>(po + job * slot_outputs(G, HD) + (size_t)e * 4),
                                         (unsigned long long)__float_as_uint(v0) | ((unsigned long long)__float_as_uint(v1) << 32));
                                if (dd == 0) st_agent(reinterpret_cast<unsigned long long*>(pml + job * SLOT_SUMS + qi * 8),
                                                      (unsigned long long)__float_as_uint(top) | ((unsigned long long)__float_as_uint(sum) << 32));
                            }
                        }
                        stores_done();
                        s.added();
                        if (job + n < jobs) s.meet();                // (what is in LDS has been read)
                    }
                    kind = O;
                } else {
                    const bool pair = kind == O || kind == DOWN;
                    const bf16_t* act = reinterpret_cast<const bf16_t*>(base + (kind == O ? P->off.at : kind == GATE_UP ? P->off.a2
                                                                                : kind == DOWN ? P->off.h : P->off.a));
                    const int count = P->kinds[kind].items, frags = P->kinds[kind].units >> (pair ? 0 : 1);
                    wait_word(words, W_GO, ++begun_phases);
                    if (word_at(words + W_STOP * 4)) break;
                    if (pair) s.product<NF_FF, true>(act, count, frags, M);
                    else s.product<NF_D, false>(act, count, frags, M);
                    if (kind == HEAD) break;
                    if (kind == DOWN) ++l;
                    kind = kind == QKV ? ATTEND : kind == O ? GATE_UP : kind == GATE_UP ? DOWN : l == P->L ? HEAD : QKV;
                }
            }
        } else {
            // The control wave: lane 8 m + j has row m and the item's column j.
            const int m = lane >> 3, j = lane & 7;
            const bool live = m < M;
            const int half = HD / 2, page = 16;
            const int pos = live ? again(A)->positions[m] : 0, b = live ? misc[W_ROW + m] : -1;
            const int blk = b >= 0 ? again(A)->blocks[(size_t)b * again(A)->max_blocks + pos / page] : -1, slot = pos % page;
            unsigned target = 0;
            int sums = 0, kind = EMBED, l = 0, begun_phases = 0;
            float w0 = 0.f, w1 = 0.f, c0 = 1.f, s0 = 0.f, c1 = 1.f, s1 = 0.f;
            float* xs = reinterpret_cast<float*>(lds + L_X);
            int id = live ? again(A)->ids[m] : -1;
            if (live && id < 0 && again(A)->device_tokens) id = again(A)->device_tokens[-1 - id];
#pragma unroll 1
            for (;;) {
                const Args P = again(A);
                char* base = P->scratch + (size_t)l * P->layer_bytes;
                const int d = P->d, ff = P->ff;
                const bool residual = kind == O || kind == DOWN || kind == EMBED;      // (the embedding is dealt as o and down are)
                const int count = kind <= HEAD ? P->kinds[kind].items : kind == EMBED ? P->kinds[O].items : 0;
                // where the items' results go, and the partial sums of squares they are scaled by
                char* to = kind == DOWN ? base + P->layer_bytes : base;
                bf16_t* out = reinterpret_cast<bf16_t*>(to + (kind == O ? P->off.a2 : kind == GATE_UP ? P->off.h : kind == QKV ? P->off.q : P->off.a));
                float* out_ssq = reinterpret_cast<float*>(to + (kind == O ? P->off.ssq2 : P->off.ssq));
                const float* ssq = reinterpret_cast<const float*>(base + (kind == GATE_UP ? P->off.ssq2 : P->off.ssq)) + (size_t)m * (d / 8) + j * 4;
                const float eps = eps_at(P, kind == GATE_UP ? 2 * l + 1 : 2 * l);
                // What the ends of this block's first two items need beside the sums is asked for long before: the weights of the norm behind o and down a phase
                // ahead; the rest of the items' as they come.  (Cosines and sines are the same for all layers.)
                float* x = P->x;
                bf16_t* kc = P->kc + (size_t)l * P->k_layer + (size_t)max(blk, 0) * Hkv * (page * HD) + (size_t)slot * HD;
                bf16_t* vc = P->vc + (size_t)l * P->v_layer + (size_t)max(blk, 0) * Hkv * (page * HD) + slot;
                float* logits = P->logits + (size_t)m * P->ld_logits + j;
                const void* w_next = norm_at(P, kind == O || kind == QKV ? 2 * l + 1 : kind == DOWN || kind == GATE_UP ? 2 * l + 2 : 0);
                if (kind == QKV || kind == GATE_UP) {
                    const int rows = P->kinds[O].items;
                    if (rank < rows) w0 = norm_weight(P, w_next, rank * 8 + j);
                    if (rank + n < rows) w1 = norm_weight(P, w_next, (rank + n) * 8 + j);
                }
                auto turn_of = [&](int item, float& c, float& sn) {
                    const size_t fi = (size_t)pos * half + 8 * (item % (HD / 16)) + j;
                    c = P->cos_t[fi];
                    sn = P->sin_t[fi];
                };
                if (kind == EMBED && b >= 0) {
                    if (rank < P->kinds[QKV].items) turn_of(rank, c0, s0);
                    if (rank + n < P->kinds[QKV].items) turn_of(rank + n, c1, s1);
                }
                if (kind != EMBED) {
                    if (!all_done(P, target, lane, begun) || word_at(words + W_STOP * 4)) {
                        set_word(words + W_STOP * 4, 1);
                        given_up = true;
                    }
                    set_word(words + W_GO * 4, ++begun_phases);
                    if (given_up) break;
                }
                if (kind == ATTEND) {
#pragma unroll 1
                    for (int job = rank; job < jobs; job += n) {
                        wait_word(words, W_SUMS + (sums & 1), (sums / 2 + 1) * WAVES);
                        ++sums;
                        set_word(words + W_FINISHED * 4, sums);
                        int part, parts;
                        const int row = row_of(job, part, parts), g = job % Hkv;
                        if (parts == 1) continue;
                        // whoever leaves the last part of a row's keys merges them all
                        unsigned before = 0;
                        if (lane == 0) before = add_agent(ctl + C_PAIRS * 32 + (row * Hkv + g) * PAIR_WORDS, 1u);
                        if (__builtin_amdgcn_readfirstlane((int)before) != (l + 1) * parts - 1) continue;
                        asm volatile("" ::: "memory");
                        merge<HD>(base + P->off.po, base + P->off.pml, job - part * Hkv, Hkv, parts, G,
                                  reinterpret_cast<bf16_t*>(base + P->off.at) + (size_t)row * q_dim + (size_t)g * G * HD, lane);
                    }
                }
                float rs = 1.f;
                if (rank < count && (kind == QKV || kind == GATE_UP || kind == HEAD)) {
                    // rsqrt(mean of the row's squares + eps): the eight lanes of a row add its partial sums up
                    float sum = 0.f;
                    if (live) {
#pragma unroll 4
                        for (int i = 0; i < d / 256; ++i) {
                            const float4 v = *reinterpret_cast<const float4*>(ssq + i * 32);
                            sum += (v.x + v.y) + (v.z + v.w);
                        }
                    }
                    sum = sum_of_eight(sum);
                    rs = rsqrtf(sum * (1.f / (float)d) + eps);
                }
#pragma unroll 1
                for (int item = rank, nth = 0; item < count; item += n, ++nth) {
                    float v1 = 0.f, v2 = 0.f, x_own = 0.f;
                    if (kind != EMBED) {
                        wait_word(words, W_SUMS + (sums & 1), (sums / 2 + 1) * WAVES);
                        const float* part = red + (sums & 1) * WAVES * 128 + j * 8 + m;
#pragma unroll
                        for (int w = 0; w < WAVES; ++w) v1 += part[w * 128];
                        if (!residual) {
#pragma unroll
                            for (int w = 0; w < WAVES; ++w) v2 += part[w * 128 + 64];
                        }
                        if (residual && nth < X_ITEMS) x_own = xs[nth * 64 + lane];
                        ++sums;
                    }
                    v1 *= rs; v2 *= rs;
                    if (residual) {
                        // eight columns of the residual stream are whole: what the product behind the next norm reads
                        float v = v1;
                        if (kind == EMBED) { if (id >= 0 && id < P->V) v = bf16_to_f32(P->table[(size_t)id * d + item * 8 + j]); }
                        else v += nth < X_ITEMS ? x_own : x[(size_t)item * 64 + lane];
                        if (nth < X_ITEMS) xs[nth * 64 + lane] = v;
                        else x[(size_t)item * 64 + lane] = v;
                        const float w = kind == EMBED || nth > 1 ? norm_weight(P, w_next, item * 8 + j) : nth ? w1 : w0;
                        store_pair(out + (size_t)m * d + item * 8 + j, v * w, live, lane);
                        const float sq = sum_of_eight(live ? v * v : 0.f);
                        if (live && j == 0) st_agent(out_ssq + (size_t)m * (d / 8) + item, sq);
                    } else if (kind == GATE_UP) {
                        store_pair(out + (size_t)m * ff + item * 8 + j, v1 / (1.f + __expf(-v1)) * v2, live, lane);
                    } else if (kind == QKV) {
                        // rotated, to the queries' buffer and the cache
                        const int head = item / (HD / 16), fi = 8 * (item % (HD / 16)) + j;
                        if (head < H + Hkv) {
                            float c = nth ? c1 : c0, sn = nth ? s1 : s0;
                            if (nth > 1 && b >= 0) turn_of(item, c, sn);
                            const float r1 = v1 * c - v2 * sn, r2 = v1 * sn + v2 * c;
                            const bool keep = b >= 0 && (head < H || blk >= 0);
                            bf16_t* dst = head < H ? out + (size_t)m * q_dim + head * HD
                                                   : kc + (size_t)(head - H) * (page * HD);
                            store_pair(dst + fi, r1, keep, lane);
                            store_pair(dst + half + fi, r2, keep, lane);
                        } else if (b >= 0 && blk >= 0) {
                            bf16_t* dst = vc + (size_t)(head - H - Hkv) * (page * HD);
                            st_agent(dst + (size_t)fi * page, f32_to_bf16(v1));
                            st_agent(dst + (size_t)(half + fi) * page, f32_to_bf16(v2));
                        }
                    } else if (live) {                            // the head
                        float* dst = logits + (size_t)item * 16;
                        dst[0] = v1;
                        dst[8] = v2;
                    }
                    if (kind != EMBED) set_word(words + W_FINISHED * 4, sums);
                }
                if (kind == HEAD) {
                    given_up = word_at(words + W_STOP * 4) != 0;
                    break;
                }
                // done: what this block has left is where everyone sees it
                const int all = kind == ATTEND ? jobs : count;
                if (rank < all) {
                    stores_done();
                    if (lane == 0) add_agent(ctl + (C_DONE + shard) * 32, 1u);
                }
                target += min(n, all);
                if (kind == DOWN) ++l;
                kind = kind == EMBED ? QKV : kind == QKV ? ATTEND : kind == ATTEND ? O : kind == O ? GATE_UP
                     : kind == GATE_UP ? DOWN : l == P->L ? HEAD : QKV;
            }
        }
    }
    if (given_up) {
        if (lane == 0) __hip_atomic_store(again(A)->gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        for (int r = 0; r < again(A)->M; ++r)
            for (int i = lane; i < again(A)->V; i += 64) again(A)->logits[(size_t)r * again(A)->ld_logits + i] = NAN;
    }
    // The last block to leave makes the control words zero again (all have read what they wanted of them).
    if (wave == CONTROL) {
        unsigned last = 0;
        if (lane == 0 && add_agent(ctl + (C_LEFT + shard) * 32, 1u) == gridDim.x / 8 - 1) last = add_agent(ctl + C_ALL_LEFT * 32, 1u) == 7 ? 1u : 0u;
        if (__builtin_amdgcn_readfirstlane((int)last)) {
            if (lane < C_PAIRS) st_agent(ctl + lane * 32, 0u);
            if (lane < 9) st_agent(ctl + C_MEMBERS * 32 + lane, 0u);
            for (int i = lane; i < MOST_PAIRS; i += 64) st_agent(ctl + C_PAIRS * 32 + i * PAIR_WORDS, 0u);
        }
    }
}

template <int HD, int NF_D, int NF_FF>
int launch_stack(const StackArgs& A, int grid, hipStream_t stream) {
    auto kernel = decode_stack_kernel<HD, NF_D, NF_FF>;
    static std::mutex mu;
    static bool asked[64] = {};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    RI_REQUIRE(e == hipSuccess && dev >= 0 && dev < 64, "ri_decode_stack: no current device: %s", hipGetErrorString(e));
    {
        std::lock_guard<std::mutex> lock(mu);
        if (!asked[dev]) {
            e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, L_BYTES);
            RI_REQUIRE(e == hipSuccess, "ri_decode_stack: %d bytes of LDS refused: %s", L_BYTES, hipGetErrorString(e));
            asked[dev] = true;
        }
    }
    kernel<<<grid, THREADS, L_BYTES, stream>>>(A);
    RI_LAUNCHED("ri_decode_stack");
    return 0;
}

// blocks that take part: one a compute unit, a multiple of eight
int stack_blocks() {
    int dev = 0, cu = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    return cu / 8 * 8;
}
// Control blocks, a launch's at a time: of uncached memory, which is never freed (memory of that kind has to stay once a kernel has read
// it), so a device has one stretch of MOST_BLOCKS, made when the first is taken.  A block belongs to whoever took it until it is given back.
constexpr int MOST_BLOCKS = 64, BLOCK_BYTES = 16 * 1024;
static_assert(CONTROL_WORDS * 4 <= BLOCK_BYTES, "a control block");
// With each goes a word of pinned host memory, likewise never freed, that a launch sets which gives up.
struct ControlBlocks { char* base = nullptr; unsigned* words = nullptr; bool refused = false, out[MOST_BLOCKS] = {}; };
constexpr int WORD_STEP = 32;                            // a line each
std::mutex control_mutex;
ControlBlocks control_blocks[64];

}  // namespace

// A control block of zeros on the current device and its word (0) on the host, or null in *block if none is to be had: all are taken, or the memory for them is
// refused (which is said once, and not asked for again).  Waits for the device: not under capture.
extern "C" int ri_decode_stack_take_control(void** block, unsigned** gave_up) {
    RI_REQUIRE(block && gave_up, "ri_decode_stack_take_control: null pointer");
    *block = nullptr;
    *gave_up = nullptr;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || dev < 0 || dev >= 64) {
        (void)hipGetLastError();
        return 0;
    }
    std::lock_guard<std::mutex> lock(control_mutex);
    ControlBlocks& c = control_blocks[dev];
    if (c.refused) return 0;
    if (!c.base) {
        void *base = nullptr, *words = nullptr;
        e = hipHostMalloc(&words, (size_t)MOST_BLOCKS * WORD_STEP * 4, hipHostMallocPortable);
        if (e == hipSuccess) e = hipExtMallocWithFlags(&base, (size_t)MOST_BLOCKS * BLOCK_BYTES, hipDeviceMallocUncached);
        if (e != hipSuccess) {
            if (words) (void)hipHostFree(words);
            (void)hipGetLastError();
            c.refused = true;
            fprintf(stderr, "[rustinfer_amd] decoding steps run part by part, not in one launch: %d bytes for their control blocks refused (%s)\n",
                    MOST_BLOCKS * BLOCK_BYTES, hipGetErrorString(e));
            return 0;
        }
        c.base = (char*)base;
        c.words = (unsigned*)words;
    }
    for (int i = 0; i < MOST_BLOCKS; ++i) {
        if (c.out[i]) continue;
        // (a launch of the one who gave it back may still be under way)
        e = hipDeviceSynchronize();
        if (e == hipSuccess) e = hipMemset(c.base + (size_t)i * BLOCK_BYTES, 0, BLOCK_BYTES);
        if (e == hipSuccess) e = hipDeviceSynchronize();
        RI_REQUIRE(e == hipSuccess, "ri_decode_stack_take_control: %s", hipGetErrorString(e));
        c.out[i] = true;
        c.words[i * WORD_STEP] = 0;
        *gave_up = c.words + i * WORD_STEP;
        *block = c.base + (size_t)i * BLOCK_BYTES;
        return 0;
    }
    return 0;
}
// Gives a block back: no launch with it follows.
extern "C" int ri_decode_stack_give_control(void* block) {
    std::lock_guard<std::mutex> lock(control_mutex);
    for (ControlBlocks& c : control_blocks) {
        const ptrdiff_t at = c.base ? (char*)block - c.base : -1;
        if (at < 0 || at >= (ptrdiff_t)MOST_BLOCKS * BLOCK_BYTES || at % BLOCK_BYTES || !c.out[at / BLOCK_BYTES]) continue;
        c.out[at / BLOCK_BYTES] = false;
        return 0;
    }
    return ri_fail("ri_decode_stack_give_control: not a block that has been taken");
}

// Whether a step of M single tokens of such a stack goes in one launch: what the kernel holds in registers and LDS, whole steps of K for every
// reader.  (Whether it pays depends on the cached tokens too: ops.decode_stack_pays.)
extern "C" int ri_decode_stack_takes(int M, int d, int ff, int H, int Hkv, int hd, int page, int V) {
    return M >= 1 && M <= MAX_ROWS && (hd == 64 || hd == 128) && page == 16 && Hkv >= 1 && M * Hkv <= MOST_PAIRS && H >= 1 && H % Hkv == 0
        && H / Hkv <= 16 && H / Hkv * hd <= ATT_VALUES && d >= 512 && d % 512 == 0 && d <= 8192 && H * hd % 512 == 0 && H * hd <= 8192
        && ff >= 512 && ff % 512 == 0 && ff <= 14336 && V % 16 == 0 && V > 0;
}
// Where slot `slot` of the parts of rows lies in a layer's stretch, with `blocks` of them: from[0], to[0] its outputs, from[1], to[1] its maxima and sums, in
// bytes; *line: what two slots may not share.
extern "C" void ri_decode_stack_slot(int M, int d, int ff, int H, int Hkv, int hd, int blocks, int slot, size_t* from, size_t* to, size_t* line) {
    const Offsets o = stack_offsets(M, d, ff, H, Hkv, hd, blocks);
    const int G = H / Hkv;
    from[0] = o.po + slot * slot_outputs(G, hd); to[0] = from[0] + (size_t)G * hd * 4;
    from[1] = o.pml + slot * SLOT_SUMS; to[1] = from[1] + (size_t)G * 8;
    *line = LINE;
}
// Entries of the model's table.
extern "C" int ri_decode_stack_table(int L) { return 4 * L + 1 + 2 * (2 * L + 1); }
// Bytes of scratch for the stretches of L layers and the one behind them, and the residual stream.
extern "C" size_t ri_decode_stack_scratch(int L, int M, int d, int ff, int H, int Hkv, int hd) {
    const int blocks = stack_blocks();
    if (blocks < 8 || M < 1 || Hkv < 1) return 0;
    return (size_t)(L + 1) * stack_offsets(M, d, ff, H, Hkv, hd, blocks).all + up256((size_t)d * MAX_ROWS * 4);
}

// model: the table of L layers on the device (ri_decode_stack_table entries, see above), the weights in tile order (q/k/v with rows in
// ri_qkv_rope_row_order).  kc, vc: the first layer's caches, k_layer and v_layer values on to the next one's.
// logits [M, ld_logits] 32-bit.  scratch: ri_decode_stack_scratch bytes, 256-byte aligned; control: a block of ri_decode_stack_take_control that no
// launch that may overlap with this one has, gave_up: its word (1 once a launch has not run to its end).  grid: blocks to launch (0: one a compute unit).
// close_us: how long the first blocks wait for the rest; join_us: and at most, where they cannot go on without; limit_us: how long for each other's results.
extern "C" int ri_decode_stack(const void* model, int L, int M, int d, int ff, int H, int Hkv, int hd, int V, int norm_dtype,
                               const int* ids, const int* device_tokens, const void* table, const int* positions, const int* row_of_token,
                               const int* kv_lens, const int* blocks, int max_blocks, const float* cos_t, const float* sin_t, void* kc, void* vc,
                               size_t k_layer, size_t v_layer, int page, float scale, float* logits, int ld_logits, void* scratch, size_t scratch_bytes,
                               unsigned* control, unsigned* gave_up, int grid, double close_us, double join_us, double limit_us, hipStream_t stream) {
    RI_REQUIRE(ri_decode_stack_takes(M, d, ff, H, Hkv, hd, page, V) && L >= 1, "ri_decode_stack: M=%d d=%d ff=%d H=%d Hkv=%d hd=%d page=%d V=%d L=%d is not taken",
               M, d, ff, H, Hkv, hd, page, V, L);
    RI_REQUIRE(model && ids && table && positions && row_of_token && kv_lens && blocks && cos_t && sin_t && kc && vc && logits
               && scratch && control && gave_up, "ri_decode_stack: null pointer");
    RI_REQUIRE(close_us >= 0 && join_us >= 0 && limit_us >= 0 && close_us <= 1e9 && join_us <= 1e9 && limit_us <= 1e9, "ri_decode_stack: bad times");
    RI_REQUIRE(ld_logits >= V && max_blocks >= 1 && (norm_dtype == RI_F32 || norm_dtype == RI_BF16), "ri_decode_stack: bad sizes or norm dtype");
    RI_REQUIRE(((uintptr_t)kc | (uintptr_t)vc) % 16 == 0 && k_layer % 8 == 0 && v_layer % 8 == 0 && (uintptr_t)scratch % 256 == 0
               && (uintptr_t)control % 128 == 0, "ri_decode_stack: unaligned pointer");
    const int all = stack_blocks();
    RI_REQUIRE(all >= 8, "ri_decode_stack: no device");
    RI_REQUIRE(grid == 0 || (grid % 8 == 0 && grid >= 8 && grid <= all), "ri_decode_stack: grid %d", grid);
    RI_REQUIRE(scratch_bytes >= ri_decode_stack_scratch(L, M, d, ff, H, Hkv, hd), "ri_decode_stack: %zu bytes of scratch are too few", scratch_bytes);
    StackArgs A;
    A.model = (const uint64_t*)model; A.L = L; A.M = M; A.d = d; A.ff = ff; A.H = H; A.Hkv = Hkv; A.V = V; A.n_f32 = norm_dtype == RI_F32;
    A.ids = ids; A.device_tokens = device_tokens; A.table = (const bf16_t*)table;
    A.positions = positions; A.row_of_token = row_of_token; A.kv_lens = kv_lens; A.blocks = blocks; A.max_blocks = max_blocks;
    A.cos_t = cos_t; A.sin_t = sin_t; A.kc = (bf16_t*)kc; A.vc = (bf16_t*)vc; A.k_layer = k_layer; A.v_layer = v_layer; A.scale = scale;
    A.logits = logits; A.ld_logits = ld_logits;
    A.off = stack_offsets(M, d, ff, H, Hkv, hd, all);
    A.layer_bytes = A.off.all;
    A.scratch = (char*)scratch;
    A.x = (float*)(A.scratch + (size_t)(L + 1) * A.layer_bytes);
    A.control = control; A.expect = all;
    A.gave_up = gave_up;
    A.close_ticks = (unsigned long long)(close_us * 100.0); A.join_ticks = (unsigned long long)(join_us * 100.0); A.limit_ticks = (unsigned long long)(limit_us * 100.0);
    if (grid == 0) grid = all;
    for (int kind = 0; kind < 5; ++kind) {
        const bool whole = kind == QKV || kind == HEAD, pair = kind == O || kind == DOWN;
        const int nks = (kind == O ? H * hd : kind == DOWN ? ff : d) / 32;
        Kind& k = A.kinds[kind];
        k.items = kind == QKV ? (H + 2 * Hkv) * hd / 16 : kind == GATE_UP ? ff / 8 : kind == HEAD ? V / 16 : d / 8;
        k.units = nks / WAVES / (pair ? 2 : 1);
        k.stride = pair ? 2048 : 1024;
        k.tile = (unsigned)nks * 1024u;
        k.second = whole ? 128u : pair ? 1024u : (unsigned)(ff / 16) * k.tile;
        k.whole = whole;
    }
    const int most_d = d > H * hd ? d : H * hd;
    if (hd == 64) {
        if (most_d <= 4096 && ff <= 8192) return launch_stack<64, 8, 16>(A, grid, stream);
        return launch_stack<64, 16, 28>(A, grid, stream);
    }
    if (most_d <= 4096 && ff <= 8192) return launch_stack<128, 8, 16>(A, grid, stream);
    if (most_d <= 4096) return launch_stack<128, 8, 28>(A, grid, stream);
    return launch_stack<128, 16, 28>(A, grid, stream);
}
