// Address rules and launch choices of the kernels as plain arithmetic, so that
// the library and a host test run the same lines (constexpr: device code too).
#pragma once
#include <algorithm>
#include <cstdint>

namespace pelica {

// Byte offset of a tile's first row, row `first` of a sequence's rows in a
// cache.  A tile that is not wanted is placed 64 rows below row 0: a
// sequence's span leaves 128 rows below 4 GiB (the check of every call), so
// modulo 2^32 each lane's piece of such a tile lies past the rows, where a
// load reads nothing.
constexpr uint32_t tile_base(bool wanted, int first, uint32_t stride_b) {
    return (uint32_t)(wanted ? first : -64) * stride_b;
}

// Positions a decode over keys [key_begin, ...) is moved up by, so that its
// first key begins a split (whole 64-key blocks): every block of it then
// starts at a row >= 0 of the range's rows, and it touches no more splits
// than its keys fill.
constexpr int range_shift(int key_begin, int split_keys) {
    return key_begin % split_keys ? split_keys - key_begin % split_keys : 0;
}

// The lane's part of the offset of load j + e of a 64-key block requested
// four loads per M0 setting: the instruction adds 1024 for each load after
// the first, which is taken off here.  Never below zero: b, the block's
// first byte, is that of a row >= 0, and step_b, the bytes from one load to
// the next, is at least 1024.
constexpr uint32_t burst_offset(uint32_t lane_off, uint32_t b, uint32_t step_b, int j, int e) {
    return lane_off + (b + (uint32_t)(j + e) * step_b - 1024u * (uint32_t)e);
}

// How an 8-wave prompt launch cuts its work: `split` 1 is one key group per
// workgroup on all of its rows (512 at head dim 64, 256 at 128); each step
// halves a workgroup's rows and doubles the number of workgroups: key groups
// 2, 4 and (head dim 64) 8, then (16) eight groups with one row tile a wave;
// at head dim 128 the last (8) is four groups of one wave, as LDS holds no
// more.  Few rows leave most CUs idle otherwise: 512 gpt-oss tokens are 64
// workgroups of 512 rows, and a full layer at position 30K took 772 us with
// 1 group, 414 with 2, 278 with 4, 317 with 8 (512 workgroups: two
// generations); 256 Qwen3 tokens over 27K keys (two rounds) 635 / 331 / 224 /
// 206; 64 gpt-oss tokens at 8K 204 / 110 / 62 / 40 / 27.5.  Where the grid
// fills the chip anyway, groups only cost: each loads its own keys (LDS writes
// beside the operand reads), and every workgroup pays its start and its merge
// (4096 fresh gpt-oss tokens 147 / 164 / 205 / 281 us).  So the split with the
// least estimated time is taken.
struct PrefillShape {
    int hd, hpk, n_kv, n_seq, T, kv_len;
    int key_begin, key_end;  // the launch's keys: a round's, or [0, kv_len)
    int window;
    bool f32;
    int64_t row_stride;
};

// us per key a group walks and us per workgroup, with most CUs idle (lat) and
// with all of them busy (thr: lower clock, shared memory rates); and us per KB
// of a workgroup's queries, and per workgroup of one group whose f16 output is
// staged in LDS.  Fitted to 1618 calls timed with every split (both
// head dims, 1-16 heads per kv head and more, 1-6000 tokens, up to 16
// sequences, windows, rounds, both query types): the choice takes 1.002x the
// best split's time in the mean, 1.06x at the 99th percentile.
struct SplitCost {
    double key_lat, wg_lat, key_thr, wg_thr;
};
constexpr SplitCost kSplitCost64[5] = {{.0245, 2.17, .0311, 5.07}, {.0238, 5.63, .0324, 7.33}, {.0262, 6.45, .038, 6.28},
                                       {.036, 5.47, .0474, 6.62}, {.0242, 3.15, .0249, 5.32}};
constexpr SplitCost kSplitCost128[4] = {{.0216, 3.18, .0263, 5.67}, {.025, 5.84, .0259, 10.7}, {.0292, 5.99, .0373, 6.86},
                                        {.0264, 4., .0259, 6.15}};
constexpr double kSplitQuery64 = .0582, kSplitQuery128 = .045, kSplitStage64 = .461, kSplitStage128 = .444;

// (of a ragged batch every sequence is taken as kv_len keys long: the lengths
// are on the GPU)
inline int prefill_split(const PrefillShape& s, int cus) {
    const bool h64 = s.hd == 64;
    const int rows = h64 ? 512 : 256, n_split = h64 ? 5 : 4;
    const int64_t same = (int64_t)s.n_kv * s.n_seq;  // blocks of one length
    // (the last share's masked tail stays inside 32-bit offsets)
    if (((int64_t)s.kv_len + 512) * s.row_stride * 2 >= (int64_t)1 << 32) return 1;
    double best = 0;
    int pick = 1;
    for (int i = 0; i < n_split; ++i) {
        const int split = 1 << i, TB = (rows >> i) / s.hpk, kg_log2 = std::min(i, h64 ? 3 : 2);
        if (TB == 0) break;
        const int n_tb = (s.T - 1) / TB + 1;
        const int64_t n = n_tb * same;
        // keys that block b (the last tokens first: the longest, as a rule)
        // walks in one key group, in whole 32-key chunks
        auto walk = [&](int b) {
            const int t0 = (n_tb - 1 - b) * TB, first = s.kv_len - s.T + t0;
            const int lo = std::max(s.window > 0 ? first + 1 - s.window : 0, s.key_begin);
            const int hi = std::min(first + std::min(TB, s.T - t0), s.key_end);
            return hi > lo ? ((hi - lo + (32 << kg_log2) - 1) >> (5 + kg_log2)) << 5 : 0;
        };
        SplitCost c = (h64 ? kSplitCost64 : kSplitCost128)[i];
        const double start = (h64 ? kSplitQuery64 : kSplitQuery128) * std::min(s.T, TB) * s.hpk * s.hd * (s.f32 ? 4 : 2) / 1024 +
                             (i == 0 && !s.f32 ? (h64 ? kSplitStage64 : kSplitStage128) : 0);
        c.wg_lat += start;
        c.wg_thr += start;
        // (a split that cannot win)
        if (i > 0 && 1.05 * (walk(0) * c.key_lat + c.wg_lat) >= best) continue;
        // running sums of the walks, over at most 16 stretches of blocks
        int step_log2 = 0;
        while (n_tb > 16 << step_log2) ++step_log2;
        const int step = 1 << step_log2, n_bin = (n_tb + step - 1) >> step_log2;
        double w[16], sums[17] = {0}, most = 0;
        for (int j = 0; j < n_bin; ++j) {
            const int b = j << step_log2, e = std::min(n_tb, b + step), first = walk(b);
            w[j] = e - b > 1 ? (first + walk(e - 1)) / 2.0 : first;
            most = std::max<double>(most, first);
            sums[j + 1] = sums[j] + w[j] * (e - b);
        }
        auto sum = [&](int b) {  // of blocks [0, b)
            const int j = b >> step_log2;
            return j < n_bin ? sums[j] + w[j] * (b - (j << step_log2)) : sums[n_bin];
        };
        const double total = sums[n_bin], mean = total / n_tb;
        // the longest block (at the clock of a chip whose CUs are busy that
        // share of the time) ...
        const double busy = most > 0 ? std::min(1.0, (double)n / cus * mean / most) : 0;
        double t = most * (c.key_lat + (c.key_thr - c.key_lat) * std::max(0.0, 2 * busy - 1)) + c.wg_lat;
        const int64_t per = n / 8, cu = std::max(1, cus / 8);
        if (n % 8 == 0 && per >= cu) {
            // An XCD gets one contiguous eighth of the blocks, in (head, block)
            // order: `full` times all of a head's blocks and a run of them, the
            // long ones or the short ones.  All the work of the XCD that gets
            // the most over its CUs ...
            const int64_t full = per / n_tb;
            const int run = (int)(per % n_tb);
            double run_most = 0;
            int run0 = 0;
            if (run > 0)
                for (int x = 0, st = 0; x < 8; ++x) {
                    const int end = st + run;
                    const double v = end <= n_tb ? sum(end) - sum(st) : total - sum(st) + sum(end - n_tb);
                    if (v > run_most) run_most = v, run0 = st;
                    st = end < n_tb ? end : end - n_tb;
                    if (st == 0) break;  // (the runs repeat)
                }
            t = std::max(t, ((full * total + run_most) * c.key_thr + per * c.wg_thr) / cu);
            // ... and g + 1 of its first g * cu + 1 blocks on one CU
            const int run1 = std::min(n_tb, run0 + run), wrapped = std::max(0, run0 + run - n_tb);
            auto count = [&](int b) {  // its blocks among the b longest
                return full * b + std::max(0, std::min(b, run1) - run0) + std::min(b, wrapped);
            };
            for (int g = 1; g <= 8 && g * cu < per; ++g) {
                int a = 0, b = n_tb;  // the fewest of the longest that are more than g * cu of its blocks
                while (a < b) {
                    const int m = (a + b) / 2;
                    if (count(m) > g * cu) b = m;
                    else a = m + 1;
                }
                t = std::max(t, (g + 1) * (walk(a - 1) * c.key_lat + c.wg_lat));
            }
        } else if (n % 8 != 0) {
            // (dealt to the XCDs in turn)
            if (n >= cus) t = std::max(t, (double)n / cus * (mean * c.key_thr + c.wg_thr));
            for (int64_t g = 1; g <= 8 && g * cus < n; ++g)
                t = std::max(t, (g + 1) * (walk((int)(g * cus / same)) * c.key_lat + c.wg_lat));
        }
        if (i == 0 || 1.05 * t < best) best = t, pick = split;
    }
    return pick;
}

}  // namespace pelica
