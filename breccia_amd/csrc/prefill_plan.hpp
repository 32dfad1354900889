// How the chunk attention kernel's work is laid out: query rows of a work-group, and the cut of page walks that
// would outlast the rest of a call.  No HIP types: host-only tests run the same functions.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <functional>
#include <numeric>
#include <vector>

#include "attn_plan.hpp"

namespace bkv {

constexpr int kPrefillPage = 16;         // cells of a page
constexpr int kPrefillRowsPerWave = 16;  // query rows
constexpr int kMaxRanges = 64;           // of one row block: the merge kernel has a lane for each

// one entry per sequence chunk
struct PrefillBatch {
    int32_t n;
    int32_t row[kMaxBatch];    // block-table row
    int32_t pos0[kMaxBatch];   // position of the chunk's first token
    int32_t n_tok[kMaxBatch];  // tokens of the chunk
    int32_t src0[kMaxBatch];   // first token row in q / out
    int32_t wg_base[kMaxBatch + 1];
};

// How a call whose longest page walks would outlast the rest is cut: the walks of an entry's
// longest blocks (its last ones) in ranges of at most pps pages, a work-group each.
struct PrefillSplit {
    int32_t pps;                       // even
    int32_t n_cut[kMaxBatch];          // row blocks of the entry that are cut
    int32_t splits[kMaxBatch];         // ranges of its longest block
    int32_t wg_base[kMaxBatch + 1];    // work-groups of the entries before; [n] = total
    int32_t unit_base[kMaxBatch + 1];  // their cut (row block, kv head) units; [n] = total
    int32_t slot_base[kMaxBatch];      // their partial results, in row blocks
};

struct PrefillPlanLimits {
    bool f16;      // the layout: f16 pools, or quantised ones
    int32_t n_kv;
    int32_t n_cu;
    int64_t rows;  // query rows a workspace holds partial results for
};

// The order in which a call's chunks are dispatched (a chunk's own blocks: longest walk first).  A chunk behind a
// long prefix has long walks only, one from scratch ends with short ones, which fill the gaps that the others leave:
// chunks go by the position a quarter into them.  Scheduled on the host, 500 random calls of 2 to 16 chunks that fill the
// chip end 6 % earlier than in the caller's order (by their last positions: 5 %), one in fifty more than 2 % later,
// by 14 % at most (one in twenty, by 29 %).  60 such calls on f16 pools, measured: 3 % sooner done than in
// the caller's order on average, 5 % later at most (by last positions: 2 % and 19 %).
enum class ChunkOrder { kByQuarter, kByEnd };
inline void order_chunks(PrefillBatch& b, int32_t n_kv, int32_t group, int32_t rows, ChunkOrder by = ChunkOrder::kByQuarter) {
    int32_t order[kMaxBatch];
    std::iota(order, order + b.n, 0);
    const auto late = [&](int32_t i) { return (by == ChunkOrder::kByQuarter ? 4 : 1) * (int64_t)b.pos0[i] + b.n_tok[i]; };
    std::stable_sort(order, order + b.n, [&](int32_t i, int32_t j) { return late(i) > late(j); });
    const PrefillBatch as_given = b;
    for (int i = 0; i < b.n; ++i) {
        b.row[i] = as_given.row[order[i]];
        b.pos0[i] = as_given.pos0[order[i]];
        b.n_tok[i] = as_given.n_tok[order[i]];
        b.src0[i] = as_given.src0[order[i]];
    }
    b.wg_base[0] = 0;
    for (int i = 0; i < b.n; ++i)
        b.wg_base[i + 1] = b.wg_base[i] + (int32_t)(((int64_t)b.n_tok[i] * group + rows - 1) / rows * n_kv);
}

// Work-groups of the fullest die if the (entry, kv head) units of an uncut call are dealt to the dies whole: with 8 or
// more, die x gets units x, x + 8, ...; with fewer, unit u is spread over dies u, u + U, ...  0 where that is too
// uneven: a die with more than a quarter over its even share, of the work-groups or of the pages they walk.  (By
// work-groups alone, a die could get the chunks with the long walks: 1.8 and 2.0 times its share of the pages cost
// such calls 1.4 and 1.5 times the time.)
constexpr int kXcds = 8;
inline int64_t even_die_share(const PrefillBatch& b, int32_t n_kv, int32_t group, int32_t rows) {
    const int units = b.n * n_kv;
    int64_t wgs[kXcds] = {}, pages[kXcds] = {}, all_wgs = 0, all_pages = 0;
    for (int u = 0; u < units; ++u) {
        const int i = u / n_kv;
        const int64_t blocks = ((int64_t)b.n_tok[i] * group + rows - 1) / rows;
        if (blocks == 0) continue;
        const int64_t walked = blocks * (2 * (int64_t)b.pos0[i] + b.n_tok[i]) / (2 * kPrefillPage) + blocks;
        const int dies = units >= kXcds ? 1 : (kXcds - u + units - 1) / units;
        all_wgs += blocks;
        all_pages += walked;
        for (int d = 0; d < dies; ++d) {
            const int x = units >= kXcds ? u % kXcds : u + d * units;
            wgs[x] += (blocks + dies - 1 - d) / dies;
            pages[x] += walked / dies;
        }
    }
    const int64_t most = *std::max_element(wgs, wgs + kXcds), most_pages = *std::max_element(pages, pages + kXcds);
    if (most * kXcds > all_wgs + all_wgs / 4 + kXcds) return 0;
    if (most_pages * kXcds > all_pages + all_pages / 4 + kXcds) return 0;
    return most;
}

// Ranges of a block that walks `pages` pages, and the (even) pages of each: evened out, none empty.
BKV_HD inline int split_ranges(int pages, int pps, int max_splits, int& each) {
    const int by_pps = (pages + pps - 1) / pps;
    const int n = by_pps < max_splits ? by_pps : max_splits;
    each = ((pages + n - 1) / n + 1) & ~1;
    return (pages + each - 1) / each;
}

// Query rows one work-group of four waves owns, in tiles of 16: two tiles a wave or one.  f16 pools: 128 when the chunks
// make more 64-row work-groups than fit the chip at two per compute unit (then sharing the page images among more rows is
// worth more than spreading out), else 64.
inline int32_t prefill_rows_per_wg(bool f16, int64_t wgs_of_64_rows, int32_t n_cu) {
    if (!f16) return 8 * kPrefillRowsPerWave;
    return wgs_of_64_rows > 2 * (int64_t)(n_cu > 0 ? n_cu : 256) ? 8 * kPrefillRowsPerWave : 4 * kPrefillRowsPerWave;
}

// When the last of the work-groups is done, in page pairs, if each unit takes the next one as it becomes free.
// runs: their pairs, in the order of dispatch.
inline int32_t last_done(const std::vector<int32_t>& runs, int32_t units) {
    const size_t at_once = std::min(runs.size(), (size_t)units);
    std::vector<int32_t> free_at(runs.begin(), runs.begin() + (ptrdiff_t)at_once);
    int32_t last = free_at.empty() ? 0 : *std::max_element(free_at.begin(), free_at.end());
    if (runs.size() == at_once) return last;
    const auto later = std::greater<int32_t>();  // a heap, the earliest in front
    std::make_heap(free_at.begin(), free_at.end(), later);
    for (size_t i = at_once; i < runs.size(); ++i) {
        std::pop_heap(free_at.begin(), free_at.end(), later);
        free_at.back() += runs[i];
        last = std::max(last, free_at.back());
        std::push_heap(free_at.begin(), free_at.end(), later);
    }
    return last;
}

// Cuts the page walks of a small call's row blocks into ranges; false where the call is better off
// uncut.  A row block's walk is a serial chain: 0.9 us a page pair on f16 pools when the compute unit
// has nothing else (2.1-2.3 us on the quantised ones, whose blocks are twice as long), and a call of a few blocks is as
// long as its longest chain while most of the chip idles (41 tokens behind 517 cells: 12 work-groups).  Cutting
// pays for a second kernel (4-9 us, by the partial rows it reads), so:
// - a call that leaves half of the compute units idle is cut if
//   - a range keeps at least 3 pairs (quantised: 2), the fixed cost of a work-group being worth several, and
//   - the chain loses 10 pairs (quantised: 5): 300 tokens behind 200 cells (16 pairs to 4) 22.9 us uncut, 22.4 cut;
//   - into one work-group per compute unit, or on f16 pools two (what fits) where a range would still be longer
//     than 8 pairs: 64 tokens behind 2000 cells 30.4 us with one, 35.0 with two; 100 behind 8000: 66.0 and 56.8
//     (append included, with eight-wave work-groups; 20.3 and 43.2 without the append now);
// - a larger call on a quantised pool (f16 pools take work-groups half as long there, two a compute unit) of up to
//   two work-groups a compute unit may be cut, into ranges of an even share of the pairs;
// - either way the chain has to lose a pair for every 32 partial results the second kernel reads; in the larger calls,
//   where the ranges come on top of a chip that is nearly busy, for every 24, and for every 20 if they don't all find a
//   compute unit at once (the chain of a cut call is then the schedule's).
// The ratios were fitted to a kernel of eight waves a work-group: a pair less gained 2.5 us (f16 1.4), a partial result cost
// 0.04 (f16 0.03), in the larger calls 0.17.  A pair is a third cheaper now and they have not been fitted again; what they do
// was measured, though: of 258 calls, random ones and those named here, on the three layouts, 107 are cut and take 0.38 of
// their time uncut on average; two of them on either quantised layout are slower for it: 60 chunks of 8 tokens behind 600
// cells, q8_0 V 38.4 uncut and 43.4 cut (int8 43.1 and 45.8), and nine unequal ones with 64 heads, 60.4 and 65.3 (64.5
// and 68.6).  What is left uncut and might pay was not looked at.
// us, uncut / cut: 41 tokens behind 517 cells 24.2 / 15.0, 100 behind 8000 249 / 43, 200 behind 3000 with q8_0 V 214 / 48,
// 300 behind 1000 on an int8 pool 103 / 39, 900 behind 2000 218 / 130; two chunks of 530 q8_0 V 48 / 39 (int8 52 / 41), 1900
// from scratch 134 / 123 (148 / 130), 400 with 48 heads 40 / 37 (44 / 38), two of 530 behind 700 92 / 87 (101 / 92).
// chain: page pairs of the cut call's longest chain, where it was worked out.
inline bool plan_prefill_split(const PrefillPlanLimits& lim, const PrefillBatch& b, int32_t rows, int32_t group, PrefillSplit& s,
                               int32_t& chain) {
    chain = 0;
    const int32_t n_kv = lim.n_kv;
    const int n_cu = lim.n_cu > 0 ? lim.n_cu : 256;
    const bool f16 = lim.f16;
    const bool idle = (int64_t)b.wg_base[b.n] * 2 <= n_cu;
    if (!idle && (f16 || b.wg_base[b.n] > 2 * n_cu)) return false;
    const int64_t least = f16 ? 3 : 2, gain = f16 ? 10 : 5;
    const int64_t room = lim.rows / rows;  // partial results the workspace holds
    int64_t work = 0;
    int32_t longest = 0;
    const auto pages_of = [&](int i, int32_t blk) {
        const int32_t last_row = std::min((blk + 1) * rows, b.n_tok[i] * group) - 1;
        return (b.pos0[i] + last_row / group) / kPrefillPage + 1;
    };
    const auto pairs_of = [&](int i, int32_t blk) { return (pages_of(i, blk) + 1) / 2; };
    const auto blocks_of = [&](int i) { return (b.n_tok[i] * group + rows - 1) / rows; };
    for (int i = 0; i < b.n; ++i) {
        const int32_t nb = blocks_of(i);
        for (int32_t k = 0; k < nb; ++k) work += (int64_t)pairs_of(i, k) * n_kv;
        if (nb) longest = std::max(longest, pairs_of(i, nb - 1));
    }
    int64_t most = std::min<int64_t>(room, n_cu);
    if (f16 && work > 8 * most) most = std::min<int64_t>(room, 2 * n_cu);
    int64_t each = std::max<int64_t>({least, (work + most - 1) / most, (longest + kMaxRanges - 1) / kMaxRanges});
    for (;; each += std::max<int64_t>(1, each / 8)) {
        if (longest < each + gain) return false;
        int64_t wgs = 0, units = 0, slots = 0;
        for (int i = 0; i < b.n; ++i) {
            const int32_t nb = blocks_of(i);
            int32_t cut = 0;
            while (cut < nb && pairs_of(i, nb - 1 - cut) > each) ++cut;
            const int64_t ranges = cut ? (pairs_of(i, nb - 1) + each - 1) / each : 1;
            s.n_cut[i] = cut;
            s.splits[i] = (int32_t)ranges;
            s.unit_base[i] = (int32_t)units;
            s.slot_base[i] = (int32_t)slots;
            s.wg_base[i] = (int32_t)wgs;
            units += (int64_t)cut * n_kv;
            slots += cut * n_kv * ranges;
            wgs += cut * n_kv * ranges + (int64_t)(nb - cut) * n_kv;
        }
        s.unit_base[b.n] = (int32_t)units;
        s.wg_base[b.n] = (int32_t)wgs;
        if (idle ? wgs <= most : slots <= room) break;
    }
    s.pps = (int32_t)each * 2;
    int64_t partials = 0;
    std::vector<int32_t> runs;  // of the work-groups, in the order of dispatch
    runs.reserve((size_t)s.wg_base[b.n]);
    for (int i = 0; i < b.n; ++i) {
        const int32_t nb = blocks_of(i);
        for (int32_t k = s.n_cut[i]; k < nb; ++k) runs.insert(runs.end(), (size_t)n_kv, pairs_of(i, nb - 1 - k));
        for (int32_t k = 0; k < s.n_cut[i]; ++k) {
            int even;
            const int pages = pages_of(i, nb - 1 - k), ranges = split_ranges(pages, s.pps, s.splits[i], even);
            partials += (int64_t)ranges * n_kv;
            for (int h = 0; h < n_kv; ++h) {
                runs.insert(runs.end(), (size_t)(ranges - 1), even / 2);
                runs.push_back((pages - (ranges - 1) * even + 1) / 2);
            }
        }
    }
    const int32_t units = f16 ? 2 * n_cu : n_cu;
    chain = last_done(runs, units);
    return (int64_t)(longest - chain) * (idle ? 32 : (int32_t)runs.size() <= units ? 24 : 20) > partials;
}

// The cut of an ordered call; in a call that nearly fills the chip its chunks go by their last positions instead where
// the schedule is shorter for it (333 tokens behind 1501, 700 behind 37 and 1021 behind 900, int8: 179 us by
// quarters, 175 by last positions).
inline bool plan_prefill(const PrefillPlanLimits& lim, PrefillBatch& b, int32_t rows, int32_t group, PrefillSplit& s) {
    int32_t chain = 0;
    bool cut = plan_prefill_split(lim, b, rows, group, s, chain);
    if (chain == 0 || (int64_t)b.wg_base[b.n] * 2 <= (lim.n_cu > 0 ? lim.n_cu : 256)) return cut;
    PrefillBatch by_end = b;
    order_chunks(by_end, lim.n_kv, group, rows, ChunkOrder::kByEnd);
    if (std::equal(b.src0, b.src0 + b.n, by_end.src0)) return cut;
    PrefillSplit other;
    int32_t shorter = 0;
    if (plan_prefill_split(lim, by_end, rows, group, other, shorter) && shorter < chain) {
        b = by_end;
        s = other;
        cut = true;
    }
    return cut;
}

}  // namespace bkv
