// Paged causal attention for chunks of many query tokens (prefill) on gfx950 matrix cores.
// The reference's counterpart is its GQA pair for T >= 16 (crates/breccia-kernels/shaders/
// qsa_attn_scores_gqa.comp, qsa_attn_apply_gqa.comp; qsa/mod.rs:116-150); the contract is the
// CPU attend (qsa/cpu.rs:197-246) with the dense selection: query token t of a chunk that
// starts at pos0 attends cells 0..pos0+t.
//
// With hundreds of query rows per kv head the work is a real matrix product (each K/V row is
// used by every query row behind it), so it goes to MFMA -- unlike the decode kernel, which
// is a GEMV per sequence.  A work-group of four waves owns 128 consecutive query rows ((token, head) pairs of one kv
// head), two tiles of 16 a wave, and walks the pages 0..page(pos) together, two at a time.  (Small calls on f16 pools:
// one tile a wave, 64 rows a work-group, two work-groups a compute unit.  Blocks that have no more than 64 rows: one tile a
// wave.)  Per page of 16 cells and per tile:
//   S^T[cell][query] = K[cell][:] . Q[query][:]        v_mfma_f32_16x16x32_f16, A = K, B = Q
//   online softmax per query (base 2), P^T in the layout S^T came out in
//   O^T[d][query]   += V^T[d][cell] . P^T[cell][query]  v_mfma_f32_16x16x32_f16 over the 32 cells of
//                                                       two pages, A = V gathered per lane (four
//                                                       cells of either page), B = P^T, high parts
//                                                       and low parts in one MFMA each
// Both products keep the per-lane query (lane % 16) fixed, so the softmax statistics never
// move between lanes, and P^T feeds the second product straight from registers.  K and V are
// exact f16; q and p are f32 values split into a high and a low f16 part (two MFMAs each), so the
// products carry ~22 significant bits and the result stays at f32-accumulate accuracy.
//
// What bounds it, and the split that follows.  Every fragment that a wave reads from LDS (1 KiB) meets the high and low
// parts of each of its tiles.  With one tile a wave that is two products, and LDS has to deliver its 128 bytes a clock
// for the matrix cores to be busy; two tiles halve it.  They need 256 registers for q and the accumulators, so a wave has
// a SIMD (512 registers) to itself: q in the upper half of the register file, which only matrix products read, everything
// else in the lower (quantised layouts: 60 to 68 values that a step needs once or not at all share the upper half).  Nobody
// fills such a wave's gaps, hence
// - a pair's scores are computed a step ahead of their softmax, whose instructions stand between those products;
// - f16 pages go from memory to LDS without passing through registers (load_to_lds);
// - every instruction counts, a wave issues one at a time (4 cycles): packed conversions, mixed-precision remainders, page
//   addresses worked out lane by lane.
// Against work-groups of eight waves with a tile each, whose steps were not pipelined (us of a call, append included): 4
// chunks of 1024 behind 2048 cells, 16 heads, f16, 332 -> 281; a prompt of 4096, 24 heads with gate, q8_0 V, 643 -> 530; three
// ragged chunks, int8, 174 -> 157; 41 tokens behind 517 cells through 12 layers 273 -> 218.  A step takes 3140 cycles on f16
// pools, 4860 with q8_0 V, 5450 with int8; its products alone would take 2048, 2560 and 3072.  On f16 pools the clock falls to
// 2.1 GHz (1200 TFLOP/s issued; registers alone, no loads, reach 1430 there): power is the next bound.  Tried on the f16 case
// and slower, 286 to 291 then: all of a step as one block, the output a step later (305); a third pair of pages in LDS (290);
// chunks of one fragment fenced off from each other (299).
// The V operand needs, per lane, four cells of one head-dim column of either page: a column of
// the row-major page image.  gfx950's transposing LDS read (ds_read_b64_tr_b16) delivers exactly
// that: within a group of 16 lanes, lane L receives element L % 4 of the 8-byte pieces that lanes
// L / 4, 4 + L / 4, 8 + L / 4 and 12 + L / 4 addressed.  With lane (c, g) addressing row 4 g + c / 4,
// halves 4 (c % 4) .. of a tile of 16 columns, lane c receives column c of the tile for cells
// 4 g .. 4 g + 3: the MFMA operand, no regrouping on the VALU.
//
// Pools with q8_0 V ([f32 scale][32 x i8] blocks, qsa_attn_apply_gqa.comp:53-77) take the same
// walk: the threads that fetch a V page dequantise it once for
// all waves, on its way into LDS, into two f16 images whose sum is the value to 22 bits
//   E[cell]    = exponent of the largest of the cell's 8 block scales (clamped to +-120),
//   a[cell][d] = code * (scale * 2^-E[cell]) = hi + lo,
// and the softmax runs over logit + E with weights exp2(logit + E - M), as in the decode kernel for
// this layout: the largest terms have weights near 1 whatever the magnitude of their values.  P.V is
// then hi.p_hi + hi.p_lo + lo.p_hi.  The denominator sums exp2(logit - R), a second exponential of its
// own: R is M until a sum comes near the end of f32's range, which rows of tiny V (E near -120) lead to.
// Int8 pools (codes with an f16 scale per 32 values, K and V alike) are dequantised the same way,
// without the exponent: both K and V become hi/lo image pairs, and the scores are
// K_hi.q_hi + K_hi.q_lo + K_lo.q_hi.  The dequantisation of the next pair stands between the P.V products of this one.
//
// A walk is a serial chain.  Where the longest of a call would outlast the rest, walks are cut into ranges, a work-group
// each, that leave partial results; prefill_merge_kernel puts them together.  Which calls, and the order of
// dispatch: prefill_plan.hpp.
#include <algorithm>
#include <type_traits>

#include "bkv_internal.hpp"
#include "gate.hpp"
#include "lane_groups.hpp"
#include "quant_decode.hpp"

namespace bkv {

namespace {

constexpr int kHd = 256;
constexpr int kPage = kPrefillPage;
constexpr int kRowsPerWave = kPrefillRowsPerWave;
constexpr int kQ8vRow = kHd / 32 * 36;  // bytes of a q8_0 row
constexpr int kI8hRow = kHd + kHd / 32 * 2;  // bytes of an int8 row: codes, then 8 f16 scales
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLoDown = 1.0f / 2048.0f;  // q's low parts enter the products times 2^11
// Two rows of a page image in LDS: 1024 bytes in one piece, as one load of a wave delivers them, and padding.  In the
// second row neighbouring 16-byte chunks (V: 32-byte pairs of them) have changed places.  With the padding, the rows
// that a read touches at a time then lie 16 (V: 32) bytes apart modulo the banks.
constexpr int kLdsRowsK = 1024 + 32;
constexpr int kLdsRowsV = 1024 + 64;

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef short tr_s4 __attribute__((__vector_size__(8)));  // what the transposing LDS read returns
typedef __attribute__((address_space(3))) tr_s4* lds_tr_ptr;
typedef const __attribute__((address_space(1))) uint8_t* page_ptr;  // said to be global memory: its address goes through integers

struct PrefillKernelParams {
    PrefillBatch b;
    const uint8_t* kpool;
    const uint8_t* vpool;
    const int32_t* tables;
    const float* q;     // [sum n_tok][n_q][256]
    const float* gate;  // optional
    float* out;         // [sum n_tok][n_q][256]
    int64_t gate_tok_stride, gate_head_stride;
    int32_t max_pages_per_seq, n_kv, n_q, group;
    float scale_log2e;
    uint32_t group_inverse, n_kv_inverse;  // floor((2^32 - 1) / n), for divided_by
    int32_t gate_in_fours;                 // four gate values can be read at once
    int32_t by_xcd;  // work-groups are dealt to the chip's 8 dies so that each die sees few (entry, kv head) units
};

// A cut call: a work-group walks one range of its block's pages and leaves a partial result,
// prefill_merge_kernel puts the ranges of a row together.
struct PrefillSplitParams : PrefillKernelParams {
    PrefillSplit s;
    float* part_o;   // [slot][row of the block][256], relative to the range's own softmax reference
    float* part_ml;  // [slot][row of the block][reference, denominator]
};

// The chip is 8 dies (XCDs), each with an L2 of its own, and work-group i runs on die i % 8.
// Every work-group of one (entry, kv head) unit walks the same K/V pages, so the dies are given
// whole units: with 8 or more units, die x serves units x, x + 8, ...; with fewer, unit u is
// served by dies u, u + U, ...  A unit's pages then stay in one die's L2 (3 MiB for a 3072-token
// chunk) instead of every die fetching every unit through the fabric.  (kXcds, and where it is done:
// prefill_plan.hpp)

// gfx950's double-depth form: 32 contraction steps, 8 halves per lane (k = 8 (lane / 16) + 0..7)
__device__ __forceinline__ f4 mfma32(h8 a, h8 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ void split_f16(float x, _Float16& hi, _Float16& lo) {
    hi = (_Float16)x;
    lo = (_Float16)(x - (float)hi);
}

// x / n and the rest, for x >= 0: the inverse is below 2^32 / n by 1 at most, so the product's quotient is right or one
// too small.  (A division by a number that only the launch knows is some 40 instructions.)
__device__ __forceinline__ int divided_by(int x, int n, uint32_t inverse, int& rest) {
    int q = (int)__umulhi((uint32_t)x, inverse);
    rest = x - q * n;
    if (rest >= n) ++q, rest -= n;
    return q;
}
__device__ __forceinline__ int divided_by(int x, int n, uint32_t inverse) {
    int rest;
    return divided_by(x, n, inverse, rest);
}

// The arguments' cache lines, asked for at once as a kernel begins: left to where each field is used, they are a chain of
// trips to memory (41 tokens behind 517 cells through 12 layers: 234 us, 218 with this and `held`).
template <typename S>
__device__ __forceinline__ void now(const PrefillBatch& b, int n_kv, const S& at_end) {
    asm volatile("" : : "s"(b.row[0]), "s"(b.pos0[0]), "s"(b.n_tok[0]), "s"(b.src0[0]), "s"(b.wg_base[0]), "s"(n_kv), "s"(at_end));
}
__device__ __forceinline__ void now(const PrefillSplit& s) {
    asm volatile("" : : "s"(s.pps), "s"(s.splits[0]), "s"(s.wg_base[0]), "s"(s.unit_base[0]), "s"(s.slot_base[0]));
}
// keeps an argument in registers from here on instead of asking for it again
template <typename T>
__device__ __forceinline__ T held(T x) {
    asm volatile("" : "+s"(x));
    return x;
}
// A pointer that came through `held` is not known to be to global memory any more: used as it is, each access is a flat one,
// which LDS counts too and which are waited for together.
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T* in_global(T* p) {
    return (__attribute__((address_space(1))) T*)p;
}

// what lane i has in x
__device__ __forceinline__ uint64_t lane_value(uint64_t x, int i) {
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)x, i);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(x >> 32), i);
    return (uint64_t)hi << 32 | lo;
}

// two f32 numbers as f16, rounded to nearest
__device__ __forceinline__ h2m to_f16(float a, float b) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    return __builtin_convertvector(f2{a, b}, h2m);
}
// x - (the f16 number hi): one v_fma_mix_f32 takes the f16 operand as it is (minus_one: -1.0f that the compiler
// cannot see through, a plain subtraction would be preceded by a conversion)
__device__ __forceinline__ float remainder_of(float x, _Float16 hi, float minus_one) {
    return __builtin_fmaf((float)hi, minus_one, x);
}
// keeps a value where it is computed: between matrix products, not behind the branch that its use stands behind
template <typename T>
__device__ __forceinline__ void stay(T& x) {
    asm volatile("" : "+v"(x));
}
// a maximum whose operands are known not to be signalling NaNs; fmaxf would quiet each of them first
__device__ __forceinline__ float max_of(float a, float b) {
    asm("v_max_f32 %0, %0, %1" : "+v"(a) : "v"(b));
    return a;
}

// 16 bytes a lane straight into LDS: lane l's go to byte lds + 16 l.  Nothing but the vector-memory count says when they
// have landed; each wave waits for its own ahead of the barrier that publishes them.
__device__ __forceinline__ void load_to_lds(unsigned lds, page_ptr base, unsigned lane_off) {
    // (the base came from a VALU instruction, which a vector-memory one must not follow closely: the copy is a scalar
    // instruction, and the wait state that m0 wants)
    uint64_t at;
    // (m0 is reserved: the compiler keeps nothing there of its own accord, and warns that it would not; what it must not do is
    // let a value that it puts there for an instruction of its own live across this)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    asm volatile("s_mov_b32 m0, %1\n\ts_mov_b64 %0, %3\n\tglobal_load_lds_dwordx4 %2, %0"
                 : "=&s"(at)
                 : "s"(lds), "v"(lane_off), "s"(base)
                 : "m0", "memory");
#pragma clang diagnostic pop
}
__device__ __forceinline__ void wait_for_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// the maximum over the four lane groups; the swaps' neighbours and wait states stand in the same block
__device__ __forceinline__ float max_over_groups(float x) {
    float a = x, b = x;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 0\n\tv_max_f32 %0, %0, %1" : "+v"(a), "+v"(b));
    b = a;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 0\n\tv_max_f32 %0, %0, %1" : "+v"(a), "+v"(b));
    return a;
}

// What a thread carries of one pair of quantised pages between its fetch and its deposit into LDS: of row tid / 16,
// block tid / 2 % 8, the codes of two 16-byte chunks of the f16 images.
struct CodeStage {
    uint2 c[2][2];                 // [page][chunk]
    unsigned scale[2];             // q8_0: the f32
    unsigned short half_scale[2];  // int8 pools: the f16's bits.  (As 32 bits they would be widened, and waited for, where
                                   // they were requested)
};

template <int LAY>
struct PrefillLds {
    // [pair of pages][page][image][pair of rows][...]: K (int8 pools: K high parts, K low parts) and V (quantised
    // pools: V high parts, V low parts)
    uint8_t kimg[2][2][LAY == BKV_LAYOUT_I8H ? 2 : 1][kPage / 2][kLdsRowsK];
    uint8_t vimg[2][2][LAY == BKV_LAYOUT_F16 ? 1 : 2][kPage / 2][kLdsRowsV];
    float e[LAY == BKV_LAYOUT_Q8V ? 2 : 1][2][kPage];  // q8_0 V: E of the cells
};
// The waves' tiles of outputs on their way to memory; rows 16 bytes apart in the banks.
constexpr int kOutRow = kHd + 4;
struct OutLds {
    float row[4][kRowsPerWave][kOutRow];
};
// byte of 16-byte chunk `chunk` of row `row` in a page image
__device__ __forceinline__ int k_at(int row, int chunk) { return (row >> 1) * kLdsRowsK + (row & 1) * 512 + (chunk ^ (row & 1)) * 16; }
__device__ __forceinline__ int v_at(int row, int chunk) { return (row >> 1) * kLdsRowsV + (row & 1) * 512 + (chunk ^ 2 * (row & 1)) * 16; }

// A row block's walk, or one range of it, by the four waves of a work-group.  TILES: tiles of 16 query rows a wave owns, the
// block's rows dealt to the waves in order.  WG_ROWS: rows of a full block, 64 per tile or more.
template <int LAY, int TILES, int WG_ROWS, bool SPLIT>
__device__ __forceinline__ void walk_block(const std::conditional_t<SPLIT, PrefillSplitParams, PrefillKernelParams>& P,
                                           PrefillLds<LAY>& L, int e, int kvh, int idx, int rb, int range, bool cut) {
    constexpr bool Q8V = LAY == BKV_LAYOUT_Q8V;
    constexpr bool I8H = LAY == BKV_LAYOUT_I8H;
    constexpr bool WIDE = LAY != BKV_LAYOUT_F16;  // V (int8 pools: K too) as two f16 images
    constexpr int kRows = kRowsPerWave * TILES;
    constexpr int kRowsPerWg = WG_ROWS;
    const int n_rows = P.b.n_tok[e] * P.group;  // query rows of this kv head
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int c = lane & 15;  // query row of the tile / cell of the page / output column group
    const int g = lane >> 4;  // which quarter of the contraction index this lane feeds
    const int row0 = rb * kRowsPerWg + wave * kRows;
    // q and the outputs pass through LDS between memory and the lanes (where not, and why: there)
    constexpr bool kStaged = LAY == BKV_LAYOUT_F16 && TILES == 1;
    const bool wave_live = row0 < n_rows;

    // pages the work-group walks: those of its last row
    const int wg_last_row = min(rb * kRowsPerWg + kRowsPerWg, n_rows) - 1;
    const int wg_pos_max = P.b.pos0[e] + divided_by(wg_last_row, P.group, P.group_inverse);
    int wg_pages = wg_pos_max / kPage + 1;
    int first_pg = 0;
    if constexpr (SPLIT) {
        if (cut) {
            int each;
            const int ranges = split_ranges(wg_pages, P.s.pps, P.s.splits[e], each);
            if (range >= ranges) return;  // the entry's longest block has more
            first_pg = range * each;
            wg_pages = min(wg_pages, first_pg + each);
        }
    }
    // this lane's query rows, and the last cell each of them attends here
    int tok[TILES], head[TILES], last_cell[TILES];
    bool row_live[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        const int row = row0 + t * kRowsPerWave + c;
        row_live[t] = row < n_rows;
        int h;
        tok[t] = divided_by(row_live[t] ? row : 0, P.group, P.group_inverse, h);
        head[t] = kvh * P.group + h;
        // a lane without a query row (past the end of the chunk) walks along with q = 0: its column of
        // the products is its own, and nothing of it is stored
        last_cell[t] = min(row_live[t] ? P.b.pos0[e] + tok[t] : 0x7fffffff, wg_pages * kPage - 1);
    }
    // Where the walk of each tile ends: behind the last page that a row of it attends.  Not later: a page may hold values
    // of V that are not finite, which a weight of 0 would not keep away from the tile's rows.  A wave that is done, or whose
    // rows lie past the chunk's end, still brings pages into LDS and joins the barriers.
    int end_pg[TILES], wave_end = 0;
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        const int first = row0 + t * kRowsPerWave, last = min(first + kRowsPerWave, n_rows) - 1;
        end_pg[t] = first < n_rows ? min((P.b.pos0[e] + divided_by(last, P.group, P.group_inverse)) / kPage + 1, wg_pages) : 0;
        wave_end = max(wave_end, end_pg[t]);
    }
    // the last cell that every row of this wave attends: pages wholly at or below it need no mask
    const int all_live = min(P.b.pos0[e] + (wave_live ? divided_by(row0, P.group, P.group_inverse) : 0), wg_pages * kPage - 1);

    constexpr int kKRow = I8H ? kI8hRow : kHd * 2;  // bytes of a row in the K pool and in the V pool
    constexpr int kVRow = I8H ? kI8hRow : Q8V ? kQ8vRow : kHd * 2;
    const size_t page_bytes = (size_t)P.n_kv * kPage * kKRow;
    const size_t head_off = (size_t)kvh * kPage * kKRow;
    const size_t v_page_bytes = (size_t)P.n_kv * kPage * kVRow;
    const size_t v_head_off = (size_t)kvh * kPage * kVRow;

    // ---- q, row by row ---------------------------------------------------------------------------
    // Lane (c, g) is to hold q[row][32 m + 8 g + 0..7], m = 0..7.  Requested like that each instruction touches 16 rows 16
    // bytes at a time, 64 cycles of the path to memory.  Requested here is a row an instruction, ahead of the table; its
    // pieces find their lanes through the memory of the V images.  41 tokens behind 517 cells through 12 layers 210 ->
    // 202 us (cycles to the first scores 8500 -> 7500).  f16 pools with one tile a wave only, whose calls may leave most of the
    // chip idle: where every compute unit asks for 128 KiB at once, memory is what q waits for (two tiles, int8, three
    // ragged chunks: 18900 cycles of prologue instead of 15700), and the quantised kernels have their walk of one tile in the
    // same kernel, whose registers came out worse for the other (158 -> 162 us).
    // (A lane without a row has the chunk's first row, and drops it.)  All of it is requested at once: behind a branch a
    // fragment, each was waited for before the next was asked for, a trip to memory each.
    const int src_q = P.b.src0[e], heads_q = P.n_q;
    f4 raw[TILES][16];
    if constexpr (kStaged) {
        const uint64_t at = (uint64_t)(uintptr_t)P.q + ((uint64_t)(src_q + tok[0]) * (uint64_t)heads_q + (uint64_t)head[0]) * (kHd * 4);
#pragma unroll
        for (int i = 0; i < 16; ++i)
            raw[0][i] = *(const __attribute__((address_space(1))) f4*)((const __attribute__((address_space(1))) float*)lane_value(at, i) + 4 * lane);
    }

    // ---- table entries, on which everything waits ----------------------------------------------------------------
    const int tid = threadIdx.x;
    const int last_pg = wg_pages - 1;
    // The table's entries come through the vector path (lane parity picks the page of a pair, past the end the last page
    // again): a scalar load among LDS reads would have to be waited for together with all of them.
    const int32_t* table = P.tables + (size_t)P.b.row[e] * (size_t)P.max_pages_per_seq;
    const auto table_pair = [&](int pg) { return table[min(pg + (lane & 1), last_pg)]; };
    const int ids_0 = table_pair(first_pg);
    int ids_v = table_pair(first_pg + 2), ids_k = table_pair(first_pg + 4);  // the pairs whose V and K are asked for next
    // addresses of a pair's pages, lane by lane as the entries came; pages are then picked from them
    const auto k_pages = [&](int ids) { return (uint64_t)(uintptr_t)(P.kpool + head_off) + (uint64_t)(unsigned)ids * (unsigned)page_bytes; };
    const auto v_pages = [&](int ids) { return (uint64_t)(uintptr_t)(P.vpool + v_head_off) + (uint64_t)(unsigned)ids * (unsigned)v_page_bytes; };
    const auto page_of = [](uint64_t pages, int w) { return (page_ptr)lane_value(pages, w); };

    // ---- pages into LDS --------------------------------------------------------------------------
    // f16 rows go there by themselves: wave w moves rows 4 w .. 4 w + 3 of a page, two rows a load; lane l delivers
    // chunk l % 32 of the image's row, which is chunk l % 32 or its neighbour of the page's row.
    const unsigned k_lane = (unsigned)(wave * 2048 + (lane >> 5) * 512 + (((lane & 31) ^ (lane >> 5)) << 4));
    const unsigned v_lane = (unsigned)(wave * 2048 + (lane >> 5) * 512 + (((lane & 31) ^ (2 * (lane >> 5))) << 4));
    const auto lds_of = [](const uint8_t* p) { return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)p; };
    const auto load_k = [&](int buf, page_ptr page, int w, int n) {
        load_to_lds(lds_of(&L.kimg[buf][w][0][2 * wave + n][0]), page, k_lane + n * 1024);
    };
    const auto load_v = [&](int buf, page_ptr page, int w, int n) {
        load_to_lds(lds_of(&L.vimg[buf][w][0][2 * wave + n][0]), page, v_lane + n * 1024);
    };
    // Quantised rows travel through registers and become high and low parts on the way.  Of its block's four chunks a
    // thread takes every other one, blocks 2, 3, 6 and 7 in the other order: eight neighbouring lanes then write eight
    // chunks that differ modulo the banks.
    const int c_row = tid >> 4, c_blk = (tid >> 1) & 7;
    const int c_chunk[2] = {4 * c_blk + (tid & 1) + (c_blk & 2), 4 * c_blk + (tid & 1) + ((c_blk & 2) ^ 2)};
    const auto fetch_codes = [&](page_ptr page, bool q8, CodeStage& st, int w) {
        const unsigned row = c_row * (q8 ? kQ8vRow : kI8hRow);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const unsigned at = q8 ? row + c_blk * 36 + 4 + (c_chunk[h] & 3) * 8 : row + c_chunk[h] * 8;
            st.c[w][h].x = *(const __attribute__((address_space(1))) unsigned*)(page + at);
            st.c[w][h].y = *(const __attribute__((address_space(1))) unsigned*)(page + (at + 4));
        }
        if (q8) st.scale[w] = *(const __attribute__((address_space(1))) unsigned*)(page + (row + c_blk * 36));
        else st.half_scale[w] = *(const __attribute__((address_space(1))) unsigned short*)(page + (row + kHd + c_blk * 2));
    };
    const auto eight = [](const h2m (&x)[4]) {
        return h8{x[0][0], x[0][1], x[1][0], x[1][1], x[2][0], x[2][1], x[3][0], x[3][1]};
    };
    // code * scale (7 + 11 significant bits) as hi = f16(code * scale) and the exact remainder (times `up`).  A scale
    // with exponent field 0 reads as zero, as everywhere.
    const auto i8h_scale = [](unsigned short bits) {
        return __builtin_bit_cast(_Float16, (unsigned short)((bits & 0x7c00u) == 0 ? 0u : bits));
    };
    const auto half_of = [&](unsigned codes, h2m s_hi, h2m s_lo, h2m* hi, h2m* lo) {
        h2m cd[2];
        codes_to_f16(codes, cd[0], cd[1]);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if constexpr (Q8V) {
                scaled_hi_lo(cd[i], s_hi, s_lo, hi[i], lo[i]);
            } else {
                hi[i] = cd[i] * s_hi;
                lo[i] = __builtin_elementwise_fma(cd[i], s_hi, -hi[i]);
            }
        }
    };
    // The deposit of a page in seven parts, which go between matrix products: the scale, then four codes at a time and the
    // stores of either chunk.
    h2m put_sh, put_sl, put_hi[4], put_lo[4];
    const auto store_parts = [&](uint8_t* to_hi, uint8_t* to_lo, int at) {
        *reinterpret_cast<h8*>(to_hi + at) = eight(put_hi);
        *reinterpret_cast<h8*>(to_lo + at) = eight(put_lo);
    };
    // the low parts of K times 2^11, like those of q: their products with q's high parts join those of q's low parts
    const auto deposit_k_part = [&](int buf, const CodeStage& st, int w, int part) {
        if (part == 0) {
            const _Float16 scale = i8h_scale(st.half_scale[w]);
            put_sh = h2m{scale, scale};
        } else if (part % 3 != 0) {
            const int h = part / 4, k = (part - 1) % 3;
            half_of(k ? st.c[w][h].y : st.c[w][h].x, put_sh, put_sl, put_hi + 2 * k, put_lo + 2 * k);
#pragma unroll
            for (int i = 2 * k; i < 2 * k + 2; ++i) put_lo[i] *= h2m{(_Float16)2048.0f, (_Float16)2048.0f};
        } else {
            store_parts(&L.kimg[buf][w][0][0][0], &L.kimg[buf][w][I8H ? 1 : 0][0][0], k_at(c_row, c_chunk[part / 3 - 1]));
        }
    };
    const auto deposit_v_part = [&](int buf, const CodeStage& st, int w, int part) {
        if (part == 0) {
            if constexpr (I8H) {
                const _Float16 scale = i8h_scale(st.half_scale[w]);
                put_sh = h2m{scale, scale};
            } else {
                // the largest scale of the row: over the lanes that differ in the block bits (1..3).  (Scales are not
                // negative: as integers their order is the same, and a NaN among foreign bytes is a large number.)
                int top = (int)(st.scale[w] & 0x7fffffffu);
                top = max(top, __builtin_amdgcn_update_dpp(0, top, 0x122, 0xf, 0xf, false));  // row_ror:2
                top = max(top, __builtin_amdgcn_update_dpp(0, top, 0x124, 0xf, 0xf, false));  // row_ror:4
                top = max(top, __builtin_amdgcn_update_dpp(0, top, 0x128, 0xf, 0xf, false));  // row_ror:8
                const int ee = min(max((top >> 23) - 127, -120), 120);
                _Float16 s_hi, s_lo;
                split_f16(__builtin_ldexpf(__builtin_bit_cast(float, st.scale[w]), -ee), s_hi, s_lo);
                put_sh = h2m{s_hi, s_hi}, put_sl = h2m{s_lo, s_lo};
                L.e[buf][w][c_row] = (float)ee;  // the same number from sixteen lanes
            }
        } else if (part % 3 != 0) {
            const int h = part / 4, k = (part - 1) % 3;
            half_of(k ? st.c[w][h].y : st.c[w][h].x, put_sh, put_sl, put_hi + 2 * k, put_lo + 2 * k);
        } else {
            store_parts(&L.vimg[buf][w][0][0][0], &L.vimg[buf][w][WIDE ? 1 : 0][0][0], v_at(c_row, c_chunk[part / 3 - 1]));
        }
    };
    constexpr int kPutParts = 7;
    const auto deposit_k = [&](int buf, const CodeStage& st, int w) {
#pragma unroll
        for (int part = 0; part < kPutParts; ++part) deposit_k_part(buf, st, w, part);
    };
    const auto deposit_v = [&](int buf, const CodeStage& st, int w) {
#pragma unroll
        for (int part = 0; part < kPutParts; ++part) deposit_v_part(buf, st, w, part);
    };
    // Rows of V past the work-group's last position were never written for these queries and may hold anything (even
    // NaN): exact zeros, before they meet a zero probability.  Each wave clears what it has put there itself; only the
    // last pair has such rows.
    const auto clear_dead_v = [&](int buf, int pg) {
        if ((pg + 2) * kPage - 1 <= wg_pos_max) return;
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const int first = min(pg + w, last_pg) * kPage;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                // f16: rows 4 w .. 4 w + 3, as loaded; quantised: two chunks, as deposited
                const int row = WIDE ? c_row : 4 * wave + 2 * j + (lane >> 5);
                const int at = v_at(row, WIDE ? c_chunk[j] : lane & 31);
                if (first + row > wg_pos_max) {
#pragma unroll
                    for (int img = 0; img < (WIDE ? 2 : 1); ++img) *reinterpret_cast<v4u*>(&L.vimg[buf][w][img][0][0] + at) = v4u{0u, 0u, 0u, 0u};
                }
            }
        }
    };

    // for the last lines of the kernel
    const float* const gate = held(P.gate);
    float* const out = held(P.out);
    const int64_t gate_tok_stride = held(P.gate_tok_stride), gate_head_stride = held(P.gate_head_stride);
    const int n_q = held(P.n_q), src0 = held(P.b.src0[e]);
    const int gate_in_fours = held(P.gate_in_fours);

    CodeStage stage_k, stage_v;
    // the first two pairs of K and the first of V; the next of either (quantised rows) in registers
    const auto load_pair_k = [&](int buf, int ids) {
        const uint64_t at = k_pages(ids);
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const page_ptr page = page_of(at, w);
            if constexpr (I8H) {
                fetch_codes(page, false, stage_k, w);
            } else {
                load_k(buf, page, w, 0);
                load_k(buf, page, w, 1);
            }
        }
    };
    const auto load_pair_v = [&](int buf, int ids) {
        const uint64_t at = v_pages(ids);
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const page_ptr page = page_of(at, w);
            if constexpr (WIDE) {
                fetch_codes(page, Q8V, stage_v, w);
            } else {
                load_v(buf, page, w, 0);
                load_v(buf, page, w, 1);
            }
        }
    };
    if constexpr (kStaged) {
        // q's rows are waited for ahead of pages that go to LDS by themselves: of those the compiler has no count, and
        // would have them arrive first
        stay(raw[0][15]);
        load_pair_k(0, ids_0);
        load_pair_k(1, ids_v);
        // eight rows of a wave at a time, as the V images have room for
        constexpr int kAtOnce = 8;
        static_assert(4 * kAtOnce * kOutRow * sizeof(float) <= sizeof(L.vimg), "q's rows in the memory of the V images");
        float* const mine = reinterpret_cast<float*>(&L.vimg) + wave * (kAtOnce * kOutRow);
        f4 q_row[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) q_row[i] = raw[0][i];
#pragma unroll
        for (int part = 0; part < 2; ++part) {
#pragma unroll
            for (int i = 0; i < kAtOnce; ++i) *reinterpret_cast<f4*>(mine + i * kOutRow + 4 * lane) = q_row[part * kAtOnce + i];
            wave_lds_fence();
            if ((c >> 3) == part) {
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    raw[0][i] = *reinterpret_cast<const f4*>(mine + (c & (kAtOnce - 1)) * kOutRow + (i >> 1) * 32 + g * 8 + (i & 1) * 4);
            }
            wave_lds_fence();
        }
    } else {
        load_pair_k(0, ids_0);
        load_pair_v(0, ids_0);
        if constexpr (!I8H) load_pair_k(1, ids_v);
        // behind the first pages' requests: q's keep the path to memory busy for 3 us
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const float* qp = P.q + ((size_t)(src0 + tok[t]) * n_q + head[t]) * kHd + g * 8;
#pragma unroll
            for (int i = 0; i < 16; ++i) raw[t][i] = *reinterpret_cast<const f4*>(qp + (i >> 1) * 32 + (i & 1) * 4);
        }
    }

    // ---- q as hi + lo f16 --------------------------------------------------------------------------
    float minus_one = -1.0f;
    asm("" : "+v"(minus_one));
    h8 qhi[TILES][8], qlo[TILES][8];
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        const float by = row_live[t] ? P.scale_log2e : 0.0f;
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            // The softmax scale (and the change to base 2) rides on q: one rounding of q, 2^-24
            // relative.  The low parts are kept times 2^11 and their products scaled back in f32
            // (kLoDown), which keeps them out of the f16 subnormals' few bits.  The product is
            // pinned as one f32 number: left to fuse it into the conversions, the compiler took the
            // remainder against f16(x * c) rounded once and stored a high part rounded twice (x * c to
            // f32, then to f16) -- two numbers that differ by an f16 ulp now and then, which showed as
            // 3e-5 in short contexts.
#pragma unroll
            for (int j = 0; j < 8; j += 2) {
                float a = raw[t][2 * m + (j >> 2)][j & 3], b = raw[t][2 * m + (j >> 2)][(j & 3) + 1];
                a = row_live[t] ? a * by : 0.0f;
                b = row_live[t] ? b * by : 0.0f;
                asm("" : "+v"(a), "+v"(b));  // the products as f32 numbers: no fusing into the conversions below
                const h2m hi = to_f16(a, b);
                const h2m lo = to_f16(remainder_of(a, hi[0], minus_one) * 2048.0f, remainder_of(b, hi[1], minus_one) * 2048.0f);
                qhi[t][m][j] = hi[0], qhi[t][m][j + 1] = hi[1];
                qlo[t][m][j] = lo[0], qlo[t][m][j + 1] = lo[1];
            }
        }
    }

    // O^T accumulators: o[tile][column tile][r] = out[row][16 (column tile) + 4 g + r]
    f4 o[TILES][16];
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int d = 0; d < 16; ++d) o[t][d] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    float m_run[TILES];  // running max of the lane's query (base-2 logits), same in all 4 g lanes
    float l_run[TILES];  // this lane's share (its 4 cells per page) of the denominator
    // q8_0 V: what l_run is relative to.  Against M its terms reach 2^(120 + kSlack) on rows of tiny V
    // (E = -120), and a few of them overflow f32; so the denominator has a reference of its own, at or
    // above M.  It leaves M when a lane's sum passes kMostL, and M meets it again from below.
    float l_ref[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) m_run[t] = l_ref[t] = -INFINITY, l_run[t] = 0.0f;
    constexpr float kMostL = 0x1p100f;

    // this lane's piece of a transposing V read: row 4 g + c / 4, halves 4 (c % 4) .. of a 16-column tile.  In odd rows
    // the even tiles have changed places with the odd ones.
    const int v_row = 4 * g + (c >> 2);
    const int v_piece = v_at(v_row, 0) + 8 * (c & 3), v_odd = 32 - 64 * (v_row & 1);
    const int k_piece = k_at(c, g);

    // scores of a pair of pages in base 2, unmasked: [tile][page][r] of cell 4 g + r, in two parts (q's high and q's
    // low parts)
    f4 s_hi[TILES][2], s_lo[TILES][2];
    // chunk i: fragment m = i % 8 of page i / 8.  K: row c, 16 bytes at element 32 m + 8 g (the same split of the head
    // dim as q): the 8 halves of a lane are the 8 contraction steps it feeds to the 32-deep MFMA
    h8 kf[16], kl[I8H ? 16 : 1];
    const auto read_k = [&](int buf, int i) {
        kf[i] = *reinterpret_cast<const h8*>(&L.kimg[buf][i >> 3][0][0][0] + k_piece + (i & 7) * 64);
        if constexpr (I8H) kl[i] = *reinterpret_cast<const h8*>(&L.kimg[buf][i >> 3][1][0][0] + k_piece + (i & 7) * 64);
    };
    const auto multiply_k = [&](int i) {
        const f4 zero = f4{0.0f, 0.0f, 0.0f, 0.0f};
        const int w = i >> 3, m = i & 7;
#pragma unroll
        for (int t = 0; t < TILES; ++t) s_hi[t][w] = mfma32(kf[i], qhi[t][m], m ? s_hi[t][w] : zero);
#pragma unroll
        for (int t = 0; t < TILES; ++t) s_lo[t][w] = mfma32(kf[i], qlo[t][m], m ? s_lo[t][w] : zero);
        if constexpr (I8H) {
#pragma unroll
            for (int t = 0; t < TILES; ++t) s_lo[t][w] = mfma32(kl[i], qhi[t][m], s_lo[t][w]);
        }
    };

    // Base-2 logits of pages pg and pg + 1 (slots 0..3: the first page's cells 4 g + r, slots 4..7: the second
    // page's), dead cells at -inf.
    float x[TILES][8];
    const auto logits = [&](int pg) {
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int r = 0; r < 8; ++r) x[t][r] = s_hi[t][r >> 2][r & 3] + s_lo[t][r >> 2][r & 3] * kLoDown;
        if ((pg + 2) * kPage - 1 > all_live) {
#pragma unroll
            for (int t = 0; t < TILES; ++t)
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    const int cell = (pg + (r >> 2)) * kPage + 4 * g + (r & 3);
                    x[t][r] = cell <= last_cell[t] ? x[t][r] : -INFINITY;
                }
        }
    };

    // Their softmax: weights as hi + lo f16, and what the accumulators have to be scaled by; in 16 parts, which go
    // between the products of the next pair's scores.
    h8 ph[TILES], pl[TILES];
    float w_[TILES][8], x_[TILES][8], pm[TILES], m_was[TILES], m_at[TILES], psum[TILES], ref[TILES], ref_at[TILES], l_new[TILES];
    bool moved[TILES];
    const auto softmax_part = [&](int buf, int part) {
        if (part == 0) {
#pragma unroll
            for (int t = 0; t < TILES; ++t) {
                // q8_0 V: the softmax runs over logit + E of the cell
#pragma unroll
                for (int r = 0; r < 8; ++r) w_[t][r] = x[t][r];
                if constexpr (Q8V) {
                    const f4 ea = *reinterpret_cast<const f4*>(&L.e[buf][0][4 * g]);
                    const f4 eb = *reinterpret_cast<const f4*>(&L.e[buf][1][4 * g]);
#pragma unroll
                    for (int r = 0; r < 4; ++r) w_[t][r] += ea[r], w_[t][r + 4] += eb[r];
                }
                pm[t] = max_of(max_of(max_of(w_[t][0], w_[t][1]), max_of(w_[t][2], w_[t][3])),
                               max_of(max_of(w_[t][4], w_[t][5]), max_of(w_[t][6], w_[t][7])));
            }
        }
        if (part == 1 || part == 2) {
            if (part - 1 < TILES) pm[part - 1] = max_over_groups(pm[part - 1]);
        }
        if (part == 3) {
#pragma unroll
            for (int t = 0; t < TILES; ++t) {
                // Cell 0 is live for every query, so from the first pair on the reference m_run is finite.
                // It follows the running maximum lazily: it moves only when a pair's maximum passes it by
                // more than kSlack (weights then reach 2^kSlack at most, far inside f16 and f32), which after
                // the first pairs is rare -- and every move costs a rescale of the 64 accumulators.  (q8_0 weights
                // multiply values of up to 2^8: products of up to 2^14, summed in f32.)
                constexpr float kSlack = 6.0f;
                moved[t] = pm[t] > m_run[t] + kSlack;  // m_run = -inf at the start: any finite maximum moves it
                m_was[t] = m_run[t];
                m_run[t] = moved[t] ? pm[t] : m_run[t];
                // a range may hold no live cell for a row (it begins past the row's position): its reference
                // stays at -inf, and the weights of its dead cells are taken against 0
                m_at[t] = SPLIT && m_run[t] == -INFINITY ? 0.0f : m_run[t];
                ref[t] = Q8V ? fmaxf(l_ref[t], m_run[t]) : m_run[t];
                ref_at[t] = SPLIT && ref[t] == -INFINITY ? 0.0f : ref[t];
                psum[t] = 0.0f;
            }
        }
        constexpr int kPairs = 4 * TILES;
        if (part >= 4 && part < 4 + kPairs) {
            const int t = (part - 4) >> 2, r0 = ((part - 4) & 3) * 2;
#pragma unroll
            for (int r = r0; r < r0 + 2; ++r) {
                w_[t][r] = __builtin_amdgcn_exp2f(w_[t][r] - m_at[t]);
                stay(w_[t][r]);
                if constexpr (Q8V) x_[t][r] = __builtin_amdgcn_exp2f(x[t][r] - ref_at[t]);
            }
        }
        if (part >= 6 && part < 6 + kPairs) {
            // p = hi + lo, both rounded to nearest (the matrix cores read f16 subnormals as the numbers
            // they are, so small weights keep their low parts' few bits)
            const int t = (part - 6) >> 2, r0 = ((part - 6) & 3) * 2;
            psum[t] += Q8V ? x_[t][r0] : w_[t][r0];
            psum[t] += Q8V ? x_[t][r0 + 1] : w_[t][r0 + 1];
            const h2m hi = to_f16(w_[t][r0], w_[t][r0 + 1]);
            const h2m lo = to_f16(remainder_of(w_[t][r0], hi[0], minus_one), remainder_of(w_[t][r0 + 1], hi[1], minus_one));
            ph[t][r0] = hi[0], ph[t][r0 + 1] = hi[1];
            pl[t][r0] = lo[0], pl[t][r0 + 1] = lo[1];
        }
        if (part == 15) {
#pragma unroll
            for (int t = 0; t < TILES; ++t) {
                l_new[t] = l_run[t] + psum[t];
                stay(ph[t]);
                stay(pl[t]);
            }
        }
    };
    const auto rescale = [&]() {
        bool any = false;
#pragma unroll
        for (int t = 0; t < TILES; ++t) any = any || moved[t] || (Q8V && l_new[t] > kMostL);
        if (__builtin_amdgcn_ballot_w64(any) != 0) {
#pragma unroll
            for (int t = 0; t < TILES; ++t) {
                const float alpha = __builtin_amdgcn_exp2f(m_was[t] - m_at[t]);  // 1, or 0 at the start
#pragma unroll
                for (int d = 0; d < 16; ++d) o[t][d] *= alpha;
                if constexpr (Q8V) {
                    l_new[t] = l_run[t] * __builtin_amdgcn_exp2f(l_ref[t] - ref_at[t]) + psum[t];
                    const float l_was = l_ref[t];
                    l_ref[t] = ref[t];
                    if (l_new[t] > kMostL) {
                        // up to the pair's largest logit (its terms are then 1 at most), and by 2^64 at least
                        float up = ref_at[t] + 64.0f;
#pragma unroll
                        for (int r = 0; r < 8; ++r) up = fmaxf(up, x[t][r]);
                        l_new[t] = 0.0f;
#pragma unroll
                        for (int r = 0; r < 8; ++r) l_new[t] += __builtin_amdgcn_exp2f(x[t][r] - up);
                        l_new[t] += l_run[t] * __builtin_amdgcn_exp2f(l_was - up);
                        l_ref[t] = up;
                    }
                } else {
                    l_new[t] = l_run[t] * alpha + psum[t];
                }
            }
        }
#pragma unroll
        for (int t = 0; t < TILES; ++t) l_run[t] = l_new[t];
    };

    // O^T += V^T . P^T over the 32 cells of the pair: per tile of 16 output columns one transposing read from either
    // page's image: lane (c, g) receives column 16 d + c of cells 4 g .. 4 g + 3 -- slots 0..3 and 4..7 of the operand,
    // the order P^T has.  Quantised V: the image of high parts meets p's high and low parts, the image of low
    // parts p's high parts.
    h8 vf[WIDE ? 32 : 16];
    const auto read_v = [&](int buf, int d) {
#pragma unroll
        for (int img = 0; img < (WIDE ? 2 : 1); ++img) {
            const int at = v_piece + (d & 1 ? v_odd : 0) + (d >> 1) * 64;
            const tr_s4 fa = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_ptr)(&L.vimg[buf][0][img][0][0] + at));
            const tr_s4 fb = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_ptr)(&L.vimg[buf][1][img][0][0] + at));
            vf[img * 16 + d] = __builtin_bit_cast(h8, __builtin_shufflevector(fa, fb, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    };
    const auto multiply_v = [&](int d, int first) {  // first: of the tiles
#pragma unroll
        for (int t = first; t < TILES; ++t) o[t][d] = mfma32(vf[d], ph[t], o[t][d]);
#pragma unroll
        for (int t = first; t < TILES; ++t) o[t][d] = mfma32(vf[d], pl[t], o[t][d]);
        if constexpr (WIDE) {
#pragma unroll
            for (int t = first; t < TILES; ++t) o[t][d] = mfma32(vf[16 + d], ph[t], o[t][d]);
        }
    };

    const auto keep_q_in_agprs = [&]() {
        if constexpr (TILES == 2) {
#pragma unroll
            for (int t = 0; t < TILES; ++t)
#pragma unroll
                for (int m = 0; m < 8; ++m) {
                    v4u a = __builtin_bit_cast(v4u, qhi[t][m]), b = __builtin_bit_cast(v4u, qlo[t][m]);
                    asm("" : "+a"(a), "+a"(b));
                    qhi[t][m] = __builtin_bit_cast(h8, a), qlo[t][m] = __builtin_bit_cast(h8, b);
                }
        }
    };
    // Fragments asked for ahead of their products, K and V, as measured with two tiles a wave (us a call, append included; what
    // counts is less the distance than the registers that it leaves): f16, 4 chunks of 1024 behind 2048 cells, 288 with 4 and 3
    // (289 with 4 and 4, 291 with 3 and 3 or 4 and 5); int8, 1204 tokens behind 495, 32 heads, 145.5 with 2 and 4 (151 with 2
    // and 5, 147 with 1 and 5, 148 with 2 and 3, 152 with 3 and 4: codes of the next pair then move through the upper half of
    // the register file, and are waited for there).  q8_0 V, a prompt of 4096, 24 heads with gate, in an earlier form of this
    // loop: 521 with 3 and 5 (525 to 535 with others).
    constexpr int kAheadK = I8H ? 2 : LAY == BKV_LAYOUT_F16 && TILES == 2 ? 4 : 3, kAheadV = I8H ? 4 : WIDE ? 5 : 3;

    if constexpr (I8H) {
        deposit_k(0, stage_k, 0);
        deposit_k(0, stage_k, 1);
        load_pair_k(1, ids_v);
    }
    if constexpr (WIDE) {
        deposit_v(0, stage_v, 0);
        deposit_v(0, stage_v, 1);
        load_pair_v(1, ids_v);
    }
    if constexpr (I8H) {
        deposit_k(1, stage_k, 0);
        deposit_k(1, stage_k, 1);
        load_pair_k(0, ids_k);
    }
    if constexpr (!I8H) wait_for_loads();
    if constexpr (!kStaged) clear_dead_v(0, first_pg);
    __syncthreads();
    if constexpr (kStaged) load_pair_v(0, ids_0);  // to where q's rows were
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        read_k(0, i);
        multiply_k(i);
    }
    if constexpr (kStaged) {
        wait_for_loads();
        clear_dead_v(0, first_pg);
    }
    __syncthreads();
    // What a step brings into LDS and requests, without products to put between
    const auto bring = [&](int pg, int buf) {
        const int ids_next = table_pair(pg + 6);
        const uint64_t k_at_pages = k_pages(ids_k), v_at_pages = v_pages(ids_v);
        if constexpr (!I8H) {
#pragma unroll
            for (int i = 0; i < 4; ++i) load_k(buf, page_of(k_at_pages, i >> 1), i >> 1, i & 1);
        }
        if constexpr (!WIDE) {
#pragma unroll
            for (int i = 0; i < 4; ++i) load_v(buf ^ 1, page_of(v_at_pages, i >> 1), i >> 1, i & 1);
        }
        ids_v = ids_k, ids_k = ids_next;
        if constexpr (I8H) {
            deposit_k(buf, stage_k, 0);
            deposit_k(buf, stage_k, 1);
            load_pair_k(0, ids_k);
        }
        if constexpr (WIDE) {
            deposit_v(buf ^ 1, stage_v, 0);
            deposit_v(buf ^ 1, stage_v, 1);
            if constexpr (Q8V) wait_for_loads();  // of K, ahead of the next codes
            load_pair_v(0, ids_v);
        }
    };
    // At the head of the step for pair j: K of pair j + 1 and V of pair j in LDS; quantised rows: K of pair j + 2 and V of
    // pair j + 1 in registers.  The step brings both into LDS, over K of pair j, whose scores are there already, and V of
    // pair j - 1.
    int pg = first_pg, buf = 0;
    const int stop = min(wg_pages - 2, end_pg[0]);
    for (; pg < stop; pg += 2, buf ^= 1) {
        keep_q_in_agprs();
#pragma unroll
        for (int i = 0; i < kAheadK; ++i) read_k(buf ^ 1, i);
        const int ids_next = table_pair(pg + 6);
        logits(pg);
        const uint64_t k_at_pages = k_pages(ids_k), v_at_pages = v_pages(ids_v);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            if (i + kAheadK < 16) read_k(buf ^ 1, i + kAheadK);
            if (!I8H && i >= 1 && i < 5) load_k(buf, page_of(k_at_pages, (i - 1) >> 1), (i - 1) >> 1, (i - 1) & 1);
            if (!WIDE && i >= 5 && i < 9) load_v(buf ^ 1, page_of(v_at_pages, (i - 5) >> 1), (i - 5) >> 1, (i - 5) & 1);
            multiply_k(i);
            if (I8H && i < 2 * kPutParts) deposit_k_part(buf, stage_k, i / kPutParts, i % kPutParts);
            softmax_part(buf, i);
        }
#pragma unroll
        for (int d = 0; d < kAheadV; ++d) read_v(buf, d);
        rescale();
        ids_v = ids_k, ids_k = ids_next;
#pragma unroll
        for (int d = 0; d < 16; ++d) {
            if (d + kAheadV < 16) read_v(buf, d + kAheadV);
            multiply_v(d, 0);
            if constexpr (WIDE) {
                if (d < 2 * kPutParts) deposit_v_part(buf ^ 1, stage_v, d / kPutParts, d % kPutParts);
                if (Q8V && d == 14) wait_for_loads();  // K of pair j + 2, asked for ahead of the scores
                if (d == 14) load_pair_v(0, ids_v);
                if (I8H && d == 1) load_pair_k(0, ids_k);  // half a step ahead of their deposit, as V's codes are
                // left to itself the scheduler does the deposit first and the products behind it
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (LAY == BKV_LAYOUT_F16) wait_for_loads();
        clear_dead_v(buf ^ 1, pg + 2);
        __syncthreads();
    }
    // Left are the walk's last pair or, where the first tile is done earlier, one that only the second tile attends (its
    // rows reach at most 16 cells further); then the work-group's other steps, without products.  A step has one barrier
    // for every wave, at its end, whichever loop the wave is in.  (With every wave in all steps: 4 chunks of 1024 behind 2048
    // cells, f16, 289 us against 292, append included; the other layouts the same: what the compiler makes of the loop above.)
    bool more = pg + 2 < wg_pages;
    if (pg < wave_end) {
        logits(pg);
#pragma unroll
        for (int i = 0; i < 16; ++i) softmax_part(buf, i);
        rescale();
        if (pg < end_pg[0]) {
#pragma unroll
            for (int d = 0; d < 16; ++d) {
                read_v(buf, d);
                multiply_v(d, 0);
            }
        } else if constexpr (TILES == 2) {
#pragma unroll
            for (int d = 0; d < 16; ++d) {
                read_v(buf, d);
                multiply_v(d, 1);
            }
        }
    }
    if (more) bring(pg, buf);
    while (more) {
        if constexpr (LAY == BKV_LAYOUT_F16) wait_for_loads();
        clear_dead_v(buf ^ 1, pg + 2);
        __syncthreads();
        pg += 2, buf ^= 1;
        more = pg + 2 < wg_pages;
        if (more) bring(pg, buf);
    }

    // ---- normalise, gate, store ---------------------------------------------------------------------
    // A lane holds 16 bytes of each 64 of its row: a store (or a request for the gate) straight from here touches 16 rows
    // 16 bytes at a time, and the path to memory takes them row by row, 64 cycles an instruction.  The wave's tile goes
    // through LDS instead (the images are done with) and leaves row by row, 1 KiB an instruction.  Cycles of the
    // epilogue, before / now: 4100 / 2900; 41 tokens behind 517 cells through 12 layers 217 -> 210 us.  f16 pools with one tile
    // a wave only: with two tiles (8300 / 6100) calls fill the chip and are at its power limit, where cycles saved
    // beside the products save no time, and the walk's registers come out worse (f16 285 against 284 us, a prompt of 4096
    // with q8_0 V 544 against 542.5).
    if constexpr (kStaged) __syncthreads();
    static_assert(sizeof(OutLds) <= sizeof(PrefillLds<LAY>), "the tiles of four waves in the memory of the images");
    float* const mine = &reinterpret_cast<OutLds*>(&L)->row[wave][0][0];
    // worked out again: the walk has no register to spare for them
    const int lane_out = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), c_out = lane_out & 15, g_out = lane_out >> 4;
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        if constexpr (Q8V) {
            // the row's four lanes to one reference, the outputs to it too (nearly always M: nothing to do)
            const float ref = max_over_lane_groups(l_ref[t]);
            const float ref_at = ref == -INFINITY ? 0.0f : ref;
            l_run[t] *= __builtin_amdgcn_exp2f(l_ref[t] - ref_at);
            if (__builtin_amdgcn_ballot_w64(m_run[t] != ref) != 0) {
                const float down = __builtin_amdgcn_exp2f(m_run[t] - ref_at);
#pragma unroll
                for (int d = 0; d < 16; ++d) o[t][d] *= down;
            }
            m_run[t] = ref;
        }
        const float l = sum_over_lane_groups(l_run[t]);
        if constexpr (!kStaged) {
            if (!row_live[t]) continue;
            if constexpr (SPLIT) {
                if (cut) {
                    const size_t slot = (size_t)P.s.slot_base[e] + (size_t)(idx * P.n_kv + kvh) * P.s.splits[e] + range;
                    const size_t at = slot * kRowsPerWg + wave * kRows + t * kRowsPerWave + c;
                    float* po = P.part_o + at * kHd + 4 * g;
#pragma unroll
                    for (int d = 0; d < 16; ++d) *reinterpret_cast<f4*>(po + 16 * d) = o[t][d];
                    if (g == 0) *reinterpret_cast<float2*>(P.part_ml + at * 2) = make_float2(m_run[t], l);
                    continue;
                }
            }
            const float inv = l > 0.0f ? 1.0f / l : 0.0f;
            const auto op = in_global(out) + ((size_t)(src0 + tok[t]) * n_q + head[t]) * kHd;
            // the gate's values in two batches of requests: one by one, each waited for before its product, they were a
            // chain of 64 trips to memory
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                f4 y[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) y[i] = o[t][half * 8 + i] * inv;
                if (gate) {
                    f4 z[8];
                    const auto at = in_global(gate) + ((size_t)(src0 + tok[t]) * gate_tok_stride + (size_t)head[t] * gate_head_stride +
                                                       128 * half + 4 * g);
                    if (gate_in_fours) {
#pragma unroll
                        for (int i = 0; i < 8; ++i) z[i] = *(const __attribute__((address_space(1))) f4*)(at + 16 * i);
                    } else {
#pragma unroll
                        for (int i = 0; i < 8; ++i)
#pragma unroll
                            for (int r = 0; r < 4; ++r) z[i][r] = at[16 * i + r];
                    }
#pragma unroll
                    for (int i = 0; i < 8; ++i)
#pragma unroll
                        for (int r = 0; r < 4; ++r) y[i][r] *= sigmoid(z[i][r]);
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) *(__attribute__((address_space(1))) f4*)(op + 16 * (half * 8 + i) + 4 * g) = y[i];
            }
        } else {
            const int live = min(n_rows - (row0 + t * kRowsPerWave), kRowsPerWave);  // rows of the tile
            if (live <= 0) continue;
            const bool parts = SPLIT && cut;
            // rows of output and gate: worked out by lane r for row r (past the chunk's end: the last row's)
            int head;
            const int row = row0 + t * kRowsPerWave + min(c_out, live - 1), tok = src0 + divided_by(row, P.group, P.group_inverse, head);
            head += kvh * P.group;
            const uint64_t out_at = (uint64_t)(uintptr_t)out + ((uint64_t)tok * (uint64_t)n_q + (uint64_t)head) * (kHd * 4);
            const uint64_t gate_at = (uint64_t)(uintptr_t)gate + (uint64_t)((int64_t)tok * gate_tok_stride + (int64_t)head * gate_head_stride) * 4;
            typedef __attribute__((address_space(1))) float* out_ptr;
            typedef const __attribute__((address_space(1))) float* gate_ptr;
            const float inv = parts ? 1.0f : l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
            for (int d = 0; d < 16; ++d) *reinterpret_cast<f4*>(mine + c_out * kOutRow + 16 * d + 4 * g_out) = o[t][d] * inv;
            wave_lds_fence();
            // from here on lane l has elements 4 l .. 4 l + 3 of every row
            const auto staged = [&](int r) { return *reinterpret_cast<const f4*>(mine + r * kOutRow + 4 * lane_out); };
            if constexpr (SPLIT) {
                if (cut) {
                    const size_t slot = (size_t)P.s.slot_base[e] + (size_t)(idx * P.n_kv + kvh) * P.s.splits[e] + range;
                    const size_t at = slot * kRowsPerWg + wave * kRows + t * kRowsPerWave;
                    float* po = P.part_o + at * kHd + 4 * lane_out;
#pragma unroll
                    for (int r = 0; r < kRowsPerWave; ++r)
                        // past the caches: what lies there when the kernel ends is written back before the merge begins.
                        // 41 tokens behind 517 cells through 12 layers 202 -> 195.5 us, longer walks the same within 1 %.  Not
                        // the quantised pools' pieces of 16 bytes: of many ranges the merge takes longer to fetch them
                        // (64 tokens behind 2000 cells, a call: q8_0 V 34.3 -> 35.8, int8 36.0 -> 38.1).
                        if (r < live) __builtin_nontemporal_store(staged(r), reinterpret_cast<f4*>(po + r * kHd));
                    if (lane_out < live) *reinterpret_cast<float2*>(P.part_ml + (at + lane_out) * 2) = make_float2(m_run[t], l);
                    continue;
                }
            }
            // the gate's values in two batches of requests: one by one, each waited for before its product, they were a
            // chain of trips to memory
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                f4 y[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) y[i] = staged(half * 8 + i);
                if (gate) {
                    f4 z[8];
                    const auto gate_row = [&](int i) { return (gate_ptr)lane_value(gate_at, half * 8 + i) + 4 * lane_out; };
                    if (gate_in_fours) {
#pragma unroll
                        for (int i = 0; i < 8; ++i) z[i] = *(const __attribute__((address_space(1))) f4*)gate_row(i);
                    } else {
#pragma unroll
                        for (int i = 0; i < 8; ++i)
#pragma unroll
                            for (int r = 0; r < 4; ++r) z[i][r] = gate_row(i)[r];
                    }
#pragma unroll
                    for (int i = 0; i < 8; ++i)
#pragma unroll
                        for (int r = 0; r < 4; ++r) y[i][r] *= sigmoid(z[i][r]);
                }
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (half * 8 + i < live) *(__attribute__((address_space(1))) f4*)((out_ptr)lane_value(out_at, half * 8 + i) + 4 * lane_out) = y[i];
            }
        }
    }
}

// SPLIT: a work-group walks one range of its block's pages and leaves a partial result.
template <int LAY, int TILES, bool SPLIT = false>
__global__ __launch_bounds__(256, TILES == 2 ? 1 : 2) void prefill_attn_kernel(
    const std::conditional_t<SPLIT, PrefillSplitParams, PrefillKernelParams> P) {
    constexpr int kRowsPerWg = 4 * TILES * kRowsPerWave;
    __shared__ __attribute__((aligned(16))) PrefillLds<LAY> L;
    now(P.b, P.n_kv, P.by_xcd);
    if constexpr (SPLIT) now(P.s);
    // ---- which (entry, kv head, block of query rows) ---------------------------------
    int e = 0, kvh, idx;  // idx: which of the unit's blocks, in dispatch order
    int range = 0;       // which range of the block's pages
    bool cut = false;    // the block is cut at all
    if constexpr (SPLIT) {
        while (e + 1 < P.b.n && (int)blockIdx.x >= P.s.wg_base[e + 1]) ++e;
        int rem = (int)blockIdx.x - P.s.wg_base[e];
        // uncut blocks first: the longest of them are longer than a range
        const int blocks = (P.b.n_tok[e] * P.group + kRowsPerWg - 1) / kRowsPerWg;
        const int uncut = (blocks - P.s.n_cut[e]) * P.n_kv;
        cut = rem >= uncut;
        if (cut) {
            rem -= uncut;
            range = rem % P.s.splits[e];
            rem /= P.s.splits[e];
        }
        idx = divided_by(rem, P.n_kv, P.n_kv_inverse, kvh) + (cut ? 0 : P.s.n_cut[e]);
    } else if (P.by_xcd) {
        const int units = P.b.n * P.n_kv;
        const int x = (int)blockIdx.x % kXcds;
        int j = (int)blockIdx.x / kXcds;
        int u;
        if (units >= kXcds) {
            u = x;
            for (;;) {
                if (u >= units) return;  // this die's share of the grid is shorter than the longest
                const int nb = (P.b.n_tok[divided_by(u, P.n_kv, P.n_kv_inverse)] * P.group + kRowsPerWg - 1) / kRowsPerWg;
                if (j < nb) break;
                j -= nb;
                u += kXcds;
            }
            idx = j;
        } else {
            u = x % units;
            const int dies = (kXcds - u + units - 1) / units;  // dies x with x % units == u
            idx = j * dies + x / units;
        }
        e = divided_by(u, P.n_kv, P.n_kv_inverse, kvh);
    } else {
        while (e + 1 < P.b.n && (int)blockIdx.x >= P.b.wg_base[e + 1]) ++e;
        const int rem = (int)blockIdx.x - P.b.wg_base[e];
        idx = divided_by(rem, P.n_kv, P.n_kv_inverse, kvh);
    }
    const int n_rows = P.b.n_tok[e] * P.group;  // query rows of this kv head
    const int n_blocks = (n_rows + kRowsPerWg - 1) / kRowsPerWg;
    if (idx >= n_blocks) return;
    // later rows attend more cells: the heaviest blocks are dispatched first
    const int rb = n_blocks - 1 - idx;
    // Few rows in a block (a short chunk, a chunk's end): a tile a wave, all four at work.  With two, half of the waves had all
    // of the products.  us of a call, two tiles / one (eight waves of one tile, before there were two): 64 chunks of 9 tokens
    // behind 2000 cells, 4 kv heads of 4 heads each, int8 167 / 129 (139), q8_0 V 139 / 118 (132); 32 chunks of 8 behind 250,
    // 2 kv heads of 8, int8 30.0 / 23.8 (26.7).
    if (TILES == 2 && n_rows - rb * kRowsPerWg <= 4 * kRowsPerWave)
        walk_block<LAY, 1, kRowsPerWg, SPLIT>(P, L, e, kvh, idx, rb, range, cut);
    else
        walk_block<LAY, TILES, kRowsPerWg, SPLIT>(P, L, e, kvh, idx, rb, range, cut);
}

// The ranges of a cut block's rows put together: one wave per row, lane d4 owns head-dim elements
// 4 d4 .. 4 d4 + 3; lane s holds range s's reference and denominator (at most 64 ranges).  Bound by
// the latency of its two trips to memory, so the partial rows are requested eight at a time before
// the references are looked at.
constexpr int kMergeWaves = 4;
constexpr int kMergeInFlight = 8;
__global__ __launch_bounds__(64 * kMergeWaves, 4) void prefill_merge_kernel(const PrefillSplitParams P, int32_t rows_per_wg) {
    now(P.b, P.n_kv, P.part_ml);
    now(P.s);
    const int w = __builtin_amdgcn_readfirstlane((int)blockIdx.x * kMergeWaves + (int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    int unit = w / rows_per_wg;
    const int r = w - unit * rows_per_wg;
    if (unit >= P.s.unit_base[P.b.n]) return;
    int e = 0;
    while (unit >= P.s.unit_base[e + 1]) ++e;
    unit -= P.s.unit_base[e];
    const int kvh = unit % P.n_kv;
    const int n_rows = P.b.n_tok[e] * P.group;
    const int rb = (n_rows + rows_per_wg - 1) / rows_per_wg - 1 - unit / P.n_kv;
    const int row = rb * rows_per_wg + r;
    if (row >= n_rows) return;
    const int wg_last_row = min(rb * rows_per_wg + rows_per_wg, n_rows) - 1;
    int each;
    const int ranges = split_ranges((P.b.pos0[e] + divided_by(wg_last_row, P.group, P.group_inverse)) / kPage + 1, P.s.pps, P.s.splits[e], each);
    const size_t at = ((size_t)P.s.slot_base[e] + (size_t)unit * P.s.splits[e]) * rows_per_wg + r;
    const float* po = P.part_o + at * kHd + 4 * lane;
    const size_t step = (size_t)rows_per_wg * kHd;
    // (past the last range its row is read again and dropped: a load behind a branch is waited for there)
    const auto part_row = [&](int i) { return *reinterpret_cast<const f4*>(po + min(i, ranges - 1) * step); };
    f4 v[kMergeInFlight];
#pragma unroll
    for (int u = 0; u < kMergeInFlight; ++u) v[u] = part_row(u);
    float2 ml = *reinterpret_cast<const float2*>(P.part_ml + (at + (size_t)min(lane, ranges - 1) * rows_per_wg) * 2);
    if (lane >= ranges) ml = make_float2(-INFINITY, 0.0f);
    int head;
    const int tok = divided_by(row, P.group, P.group_inverse, head);
    head += kvh * P.group;
    const size_t out_row = (size_t)(P.b.src0[e] + tok);
    float4 gt = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (P.gate) {
        const float* gp = P.gate + out_row * P.gate_tok_stride + (size_t)head * P.gate_head_stride + 4 * lane;
        gt = make_float4(gp[0], gp[1], gp[2], gp[3]);
    }
    // the first range holds cell 0, which every row attends: the maximum is finite
    float mx = ml.x;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
    const float wt = __builtin_amdgcn_exp2f(ml.x - mx);
    float l = wt * ml.y;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) l += __shfl_xor(l, off, 64);
    f4 acc = f4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int s = 0;;) {
#pragma unroll
        for (int u = 0; u < kMergeInFlight; ++u)
            if (s + u < ranges) acc += v[u] * __shfl(wt, s + u, 64);
        s += kMergeInFlight;
        if (s >= ranges) break;
#pragma unroll
        for (int u = 0; u < kMergeInFlight; ++u) v[u] = part_row(s + u);
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    float4 y = make_float4(acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv);
    if (P.gate) y = make_float4(y.x * sigmoid(gt.x), y.y * sigmoid(gt.y), y.z * sigmoid(gt.z), y.w * sigmoid(gt.w));
    *reinterpret_cast<float4*>(P.out + (out_row * P.n_q + head) * kHd + 4 * lane) = y;
}

template <int LAY, int TILES>
hipError_t launch_split(bkv_pool* p, const PrefillSplitParams& kp, hipStream_t stream) {
    constexpr int kRows = 4 * TILES * kRowsPerWave;
    launch_staged(p, BKV_STAGE_PREFILL_ATTN, prefill_attn_kernel<LAY, TILES, true>,
                  dim3((unsigned)kp.s.wg_base[kp.b.n]), dim3(256), 0, stream, kp);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    const unsigned rows = (unsigned)kp.s.unit_base[kp.b.n] * kRows;
    launch_staged(p, BKV_STAGE_ATTN_MERGE, prefill_merge_kernel, dim3(rows / kMergeWaves), dim3(64 * kMergeWaves), 0,
                  stream, kp, (int32_t)kRows);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_prefill_attn(bkv_pool* p, int32_t layer, const PrefillBatch& b, const AttnArgs& a,
                               int32_t rows_per_wg, const PrefillSplit* split, const ChunkWorkspace* ws, hipStream_t stream) {
    PrefillSplitParams sp;
    PrefillKernelParams& kp = sp;
    kp.b = b;
    kp.kpool = p->k_layer[(size_t)layer];
    kp.vpool = p->v_layer[(size_t)layer];
    kp.tables = p->table_dev;
    kp.q = a.q;
    kp.gate = a.gate;
    kp.out = a.out;
    kp.gate_tok_stride = a.gate_seq_stride;
    kp.gate_head_stride = a.gate_head_stride;
    kp.max_pages_per_seq = p->desc.max_pages_per_seq;
    kp.n_kv = p->g.n_kv;
    kp.n_q = a.n_q_head;
    kp.group = a.n_q_head / p->g.n_kv;
    kp.group_inverse = 0xffffffffu / (uint32_t)kp.group;
    kp.n_kv_inverse = 0xffffffffu / (uint32_t)kp.n_kv;
    kp.gate_in_fours = (((uint64_t)(uintptr_t)a.gate | (uint64_t)a.gate_seq_stride * 4 | (uint64_t)a.gate_head_stride * 4) & 15) == 0;
    kp.scale_log2e = a.scale * kLog2e;
    int32_t grid = b.wg_base[b.n];
    if (grid == 0) return hipSuccess;
    if (split) {
        kp.by_xcd = 0;
        sp.s = *split;
        sp.part_o = ws->o;
        sp.part_ml = ws->ml;
        if (p->g.layout == BKV_LAYOUT_Q8V) return launch_split<BKV_LAYOUT_Q8V, 2>(p, sp, stream);
        if (p->g.layout == BKV_LAYOUT_I8H) return launch_split<BKV_LAYOUT_I8H, 2>(p, sp, stream);
        return launch_split<BKV_LAYOUT_F16, 1>(p, sp, stream);
    }
    // Deal the work-groups to the dies by unit where that costs little: the grid then holds 8 x the
    // longest die's share, and work-groups past a shorter die's share leave at once.
    kp.by_xcd = 0;
    const int64_t share = even_die_share(b, p->g.n_kv, kp.group, rows_per_wg);
    if (share) {
        kp.by_xcd = 1;
        grid = (int32_t)(share * kXcds);
    }
    if (p->g.layout == BKV_LAYOUT_Q8V)
        launch_staged(p, BKV_STAGE_PREFILL_ATTN, prefill_attn_kernel<BKV_LAYOUT_Q8V, 2>, dim3((unsigned)grid), dim3(256), 0,
                      stream, kp);
    else if (p->g.layout == BKV_LAYOUT_I8H)
        launch_staged(p, BKV_STAGE_PREFILL_ATTN, prefill_attn_kernel<BKV_LAYOUT_I8H, 2>, dim3((unsigned)grid), dim3(256), 0,
                      stream, kp);
    else if (rows_per_wg == 8 * kRowsPerWave)
        launch_staged(p, BKV_STAGE_PREFILL_ATTN, prefill_attn_kernel<BKV_LAYOUT_F16, 2>, dim3((unsigned)grid), dim3(256), 0,
                      stream, kp);
    else
        launch_staged(p, BKV_STAGE_PREFILL_ATTN, prefill_attn_kernel<BKV_LAYOUT_F16, 1>, dim3((unsigned)grid), dim3(256), 0,
                      stream, kp);
    return hipGetLastError();
}

}  // namespace bkv
