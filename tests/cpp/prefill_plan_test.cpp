// How chunk attention cuts its page walks (breccia_amd/csrc/prefill_plan.hpp), over random batches: every cut the
// planner returns is walked the way the kernels walk it -- work-group index to (entry, row block, kv head, range), and
// row block to its partial results -- and has to cover every page of every row block once, inside the workspace.
// Prints what it met and exits 0.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <utility>
#include <vector>

#include "../../breccia_amd/csrc/prefill_plan.hpp"

using namespace bkv;

static void must(bool ok, const char* what, int at) {
    if (!ok) {
        std::fprintf(stderr, "FAILED in batch %d: %s\n", at, what);
        std::exit(1);
    }
}

// Whether the call's walks are cut: q heads over two kv heads, (cells before, tokens) of its chunks, on 256 compute units.
static bool is_cut(bool f16, int n_q, const std::vector<std::pair<int, int>>& chunks) {
    const PrefillPlanLimits lim{f16, 2, 256, 4096 * 8};
    const int group = n_q / 2;
    PrefillBatch b{};
    int64_t wgs64 = 0;
    for (const auto& c : chunks) {
        b.pos0[b.n] = c.first;
        b.n_tok[b.n++] = c.second;
        wgs64 += ((int64_t)c.second * group + 63) / 64 * lim.n_kv;
    }
    const int rows = prefill_rows_per_wg(f16, wgs64, lim.n_cu);
    order_chunks(b, lim.n_kv, group, rows);
    PrefillSplit s;
    return plan_prefill(lim, b, rows, group, s);
}

// Calls measured both ways, on either side of the planner's lines.
static void lines() {
    using Chunks = std::vector<std::pair<int, int>>;
    must(!is_cut(false, 16, Chunks(4, {0, 270})), "four chunks of 270: 38 us uncut, 52 cut", -1);
    must(!is_cut(false, 48, {{0, 600}}), "600 tokens with 48 heads: 70 us uncut, 79 cut", -1);
    must(!is_cut(false, 16, Chunks(32, {250, 8})), "32 chunks of 8 behind 250: 28 us uncut, 31 cut", -1);
    must(!is_cut(true, 16, Chunks(16, {500, 30})), "f16, 16 chunks of 30 behind 500: 35 us uncut, 38 cut", -1);
    must(is_cut(false, 16, Chunks(2, {0, 530})), "two chunks of 530: 60 us uncut, 48 cut", -1);
    must(is_cut(false, 16, {{0, 1900}}), "1900 tokens: 169 us uncut, 151 cut", -1);
    must(is_cut(false, 48, {{0, 400}}), "400 tokens with 48 heads: 51 us uncut, 45 cut", -1);
    must(is_cut(true, 16, {{517, 41}}), "f16, 41 tokens behind 517: 37 us uncut, 24 cut", -1);
}

// When an uncut call on a quantised pool ends, in page pairs, its chunks in the batch's order.
static int32_t uncut_end(const PrefillBatch& b, int group) {
    std::vector<int32_t> runs;
    for (int i = 0; i < b.n; ++i)
        for (int rb = (b.n_tok[i] * group + 127) / 128 - 1; rb >= 0; --rb) {
            const int last_row = std::min((rb + 1) * 128, b.n_tok[i] * group) - 1;
            runs.insert(runs.end(), 2, ((b.pos0[i] + last_row / group) / kPrefillPage + 2) / 2);
        }
    return last_done(runs, 256);
}

// The order of dispatch: every chunk once, with what belongs to it, and no call much worse for it.
static void order() {
    std::mt19937 rng(5);
    const auto pick = [&](int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); };
    const auto log_pick = [&](double lo, double hi) { return (int)std::lround(lo * std::pow(hi / lo, (rng() % 4096) / 4095.0)); };
    double sum = 0.0, worst = 0.0;
    int calls = 0;
    while (calls < 300) {
        PrefillBatch b{};
        b.n = pick(2, 16);
        const int group = 4 * pick(1, 4);
        int64_t wgs = 0, src = 0;
        for (int i = 0; i < b.n; ++i) {
            b.row[i] = i;
            b.n_tok[i] = log_pick(16, 3000);
            b.pos0[i] = pick(0, 1) ? log_pick(16, 6000) : 0;
            b.src0[i] = (int32_t)src;
            src += b.n_tok[i];
            wgs += ((int64_t)b.n_tok[i] * group + 127) / 128 * 2;
        }
        if (wgs < 200 || wgs > 1500) continue;
        PrefillBatch o = b;
        order_chunks(o, 2, group, 128);
        std::vector<char> seen(b.n, 0);
        for (int i = 0; i < b.n; ++i) {
            const int r = o.row[i];
            must(!seen[r]++ && o.pos0[i] == b.pos0[r] && o.n_tok[i] == b.n_tok[r] && o.src0[i] == b.src0[r], "a chunk's own values", calls);
        }
        const double ratio = (double)uncut_end(o, group) / (double)uncut_end(b, group);
        sum += ratio;
        worst = std::max(worst, ratio);
        ++calls;
    }
    std::printf("order of dispatch: %.3f of the caller's on average, %.3f at most\n", sum / calls, worst);
    must(sum / calls < 0.96 && worst < 1.16, "the order of dispatch costs more than it gains", calls);
}

// Units dealt to the dies, walked the way the kernel does it: every row block of every unit once, no die with far more
// than its share of the pages.
static void dies() {
    std::mt19937 rng(9);
    const auto pick = [&](int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); };
    const auto log_pick = [&](double lo, double hi) { return (int)std::lround(lo * std::pow(hi / lo, (rng() % 4096) / 4095.0)); };
    int dealt = 0;
    double worst = 0.0;
    for (int at = 0; at < 20000; ++at) {
        const int n_kv = 1 << pick(0, 3), group = pick(1, 16), rows = pick(0, 1) ? 64 : 128;
        PrefillBatch b{};
        b.n = pick(1, 12);
        const int tok = log_pick(1, 3000), before = log_pick(1, 8000), alike = pick(0, 1);
        for (int i = 0; i < b.n; ++i) {
            b.n_tok[i] = alike ? pick(tok / 2, tok) : pick(0, 7) ? log_pick(1, 3000) : 0;
            b.pos0[i] = alike ? before : pick(0, 1) ? log_pick(1, 8000) : 0;
        }
        const int64_t share = even_die_share(b, n_kv, group, rows);
        if (!share) continue;
        ++dealt;
        const int units = b.n * n_kv;
        const auto blocks_of = [&](int i) { return (b.n_tok[i] * group + rows - 1) / rows; };
        std::vector<std::vector<int>> seen;
        for (int u = 0; u < units; ++u) seen.push_back(std::vector<int>(blocks_of(u / n_kv), 0));
        int64_t pages[kXcds] = {}, all = 0;
        for (int64_t wg = 0; wg < share * kXcds; ++wg) {
            const int x = (int)(wg % kXcds);
            int j = (int)(wg / kXcds), u, idx;
            if (units >= kXcds) {
                for (u = x; u < units; u += kXcds) {
                    const int nb = blocks_of(u / n_kv);
                    if (j < nb) break;
                    j -= nb;
                }
                if (u >= units) continue;
                idx = j;
            } else {
                u = x % units;
                idx = j * ((kXcds - u + units - 1) / units) + x / units;
            }
            const int i = u / n_kv;
            if (idx >= blocks_of(i)) continue;
            ++seen[u][idx];
            const int last_row = std::min((blocks_of(i) - idx) * rows, b.n_tok[i] * group) - 1;
            const int walked = (b.pos0[i] + last_row / group) / kPrefillPage + 1;
            pages[x] += walked;
            all += walked;
        }
        for (const auto& unit : seen)
            for (int times : unit) must(times == 1, "a row block dealt other than once", at);
        const double most = (double)*std::max_element(pages, pages + kXcds) * kXcds / (double)std::max<int64_t>(all, 1);
        if (all > 20000) worst = std::max(worst, most);
    }
    std::printf("%d dealt to the dies, the fullest with %.2f of its share of the pages\n", dealt, worst);
    must(dealt > 1000 && worst < 1.35, "dealing to the dies", -1);
}

int main(int argc, char** argv) {
    lines();
    order();
    dies();
    std::mt19937 rng(argc > 1 ? (unsigned)std::atoi(argv[1]) : 1u);
    const int batches = argc > 2 ? std::atoi(argv[2]) : 100000;
    const auto pick = [&](int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); };
    const auto log_pick = [&](double lo, double hi) { return (int)std::lround(lo * std::pow(hi / lo, (rng() % 4096) / 4095.0)); };
    int cuts = 0, widened = 0, unbalanced = 0, most_ranges = 0;
    double fullest = 0.0;
    for (int at = 0; at < batches; ++at) {
        PrefillPlanLimits lim{};
        lim.f16 = pick(0, 1);
        lim.n_kv = 1 << pick(0, 3);
        lim.n_cu = pick(0, 3) ? 256 : pick(16, 304);
        lim.rows = 4096 * 8;
        const int group = pick(1, 16);
        PrefillBatch b{};
        b.n = pick(0, 2) ? pick(1, 3) : log_pick(1, kMaxBatch);
        const int most_tok = log_pick(1, 3000), most_before = log_pick(1, 300000);
        int64_t wgs64 = 0;
        for (int i = 0; i < b.n; ++i) {
            b.n_tok[i] = pick(0, 7) ? log_pick(1, most_tok) : 0;
            b.pos0[i] = pick(0, 2) ? log_pick(1, most_before) : 0;
            wgs64 += ((int64_t)b.n_tok[i] * group + 63) / 64 * lim.n_kv;
        }
        const int rows = prefill_rows_per_wg(lim.f16, wgs64, lim.n_cu);
        const auto blocks_of = [&](int i) { return (b.n_tok[i] * group + rows - 1) / rows; };
        order_chunks(b, lim.n_kv, group, rows);
        const int64_t wgs = b.wg_base[b.n];
        PrefillSplit s;
        if (wgs == 0 || !plan_prefill(lim, b, rows, group, s)) continue;
        ++cuts;
        const int64_t room = lim.rows / rows;
        must(s.pps > 0 && s.pps % 2 == 0, "an odd range", at);
        must(s.wg_base[0] == 0 && s.unit_base[0] == 0, "bases begin at zero", at);
        // pages of the row block `idx` of entry e, blocks counted from the last one
        const auto pages_of = [&](int e, int idx) {
            const int rb = blocks_of(e) - 1 - idx;
            const int last_row = std::min(rb * rows + rows, b.n_tok[e] * group) - 1;
            return (b.pos0[e] + last_row / group) / kPrefillPage + 1;
        };
        std::vector<std::vector<std::vector<int>>> walked(b.n);  // [entry][block, kv head] -> how often each page
        for (int e = 0; e < b.n; ++e) {
            must(s.n_cut[e] >= 0 && s.n_cut[e] <= blocks_of(e), "more blocks cut than there are", at);
            must(s.splits[e] >= 1 && s.splits[e] <= kMaxRanges, "more ranges than the merge has lanes", at);
            for (int idx = 0; idx < blocks_of(e); ++idx)
                for (int h = 0; h < lim.n_kv; ++h) walked[e].push_back(std::vector<int>(pages_of(e, idx), 0));
        }
        std::vector<char> slot_used(room, 0);
        int used = 0;
        for (int wg = 0; wg < s.wg_base[b.n]; ++wg) {
            int e = 0;
            while (e + 1 < b.n && wg >= s.wg_base[e + 1]) ++e;
            int rem = wg - s.wg_base[e], range = 0;
            const int uncut = (blocks_of(e) - s.n_cut[e]) * lim.n_kv;
            const bool cut = rem >= uncut;
            if (cut) {
                rem -= uncut;
                range = rem % s.splits[e];
                rem /= s.splits[e];
            }
            const int kvh = rem % lim.n_kv, idx = rem / lim.n_kv + (cut ? 0 : s.n_cut[e]);
            must(idx < blocks_of(e), "a work-group past the entry's blocks", at);
            const int pages = pages_of(e, idx);
            int first = 0, end = pages;
            if (cut) {
                int each;
                const int ranges = split_ranges(pages, s.pps, s.splits[e], each);
                must(ranges >= 2 && ranges <= s.splits[e] && each % 2 == 0 && each <= s.pps, "a block's ranges", at);
                most_ranges = std::max(most_ranges, ranges);
                if (range >= ranges) continue;
                first = range * each;
                end = std::min(pages, first + each);
                const int64_t slot = s.slot_base[e] + (int64_t)(idx * lim.n_kv + kvh) * s.splits[e] + range;
                must(slot >= 0 && slot < room, "a partial result outside the workspace", at);
                must(!slot_used[slot], "two ranges in one place", at);
                slot_used[slot] = 1;
                used = std::max(used, (int)slot + 1);
            }
            must(first < end, "an empty range", at);
            for (int pg = first; pg < end; ++pg) ++walked[e][(size_t)idx * lim.n_kv + kvh][pg];
        }
        for (const auto& entry : walked)
            for (const auto& block : entry)
                for (int times : block) must(times == 1, "a page is walked other than once", at);
        // the merge's units: the cut blocks, entry by entry
        for (int e = 0; e < b.n; ++e)
            must(s.unit_base[e + 1] - s.unit_base[e] == s.n_cut[e] * lim.n_kv, "units of the merge", at);
        fullest = std::max(fullest, (double)used / (double)room);
        if (lim.f16 && s.wg_base[b.n] > lim.n_cu) ++widened;
        if (wgs * 2 > lim.n_cu) ++unbalanced;
    }
    std::printf("%d cut: %d two work-groups a compute unit, %d unbalanced, up to %d ranges, workspace filled to %.3f\n", cuts, widened,
                unbalanced, most_ranges, fullest);
    // the sweep has to reach the planner's ends
    return cuts > batches / 20 && widened > 100 && unbalanced > 100 && most_ranges >= 63 && fullest > 0.99 ? 0 : 2;
}
