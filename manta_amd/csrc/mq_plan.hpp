// mq_plan.hpp -- the row ranges of a multi-query call's passes (host
// arithmetic only: no HIP types, so that it also compiles by itself).
//
// Multi-query top-k runs in passes over growing row prefixes: pass 0 keeps
// every key of its rows, and each later pass starts from the k-th best key
// of all earlier rows, so only a few times k keys per query survive a pass.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <vector>

namespace manta {

constexpr int64_t kMqSelectKeys = 16384;  // LDS keys of the select kernel

// Byte offset of the last whole word of `left` rows' f16 block scales, nb a
// row, counted from the first of them.  The q4 kernel copies scales 4 bytes
// at a time and clamps every copy to this word, so the first row's scales
// must start on a word (an even row, whatever nb), and an odd count ends half
// way through a word (the allocation is padded to one).
constexpr int mq4_scale_limit(int left, int nb) { return (left * nb * 2 - 1) & ~3; }

struct MqPass {
    int64_t begin = 0;
    int64_t end = 0;
    int64_t rows_per_wg = 0;
    int R = 0;                // workgroups over the rows
    int select_threads = 256;
    double grow = 1.0;        // rows up to its end over those before it
};

inline MqPass mq_pass(int64_t begin, int64_t end, int chunk, int groups, int64_t max_rows_per_wg, int wgs) {
    MqPass p;
    p.begin = begin;
    p.end = end;
    const int64_t chunks = (end - begin + chunk - 1) / chunk;
    int64_t R = std::max<int64_t>(1, std::min<int64_t>(chunks, std::max(1, wgs / groups)));
    int64_t cpw = (chunks + R - 1) / R;
    if (max_rows_per_wg > 0) cpw = std::max<int64_t>(1, std::min<int64_t>(cpw, max_rows_per_wg / chunk));
    p.rows_per_wg = cpw * chunk;
    p.R = (int)((chunks + cpw - 1) / cpw);
    return p;
}

// Region capacity of a top-k pass: the best k after a compaction plus one
// chunk of appends, with slack so a compaction frees at least k slots (the
// 512-query kernel needs rc >= k + 2.5 chunks: true for its chunks of 64 or
// 128 rows).
inline int mq_region_keys(int64_t k, int chunk) { return (int)(((2 * k + 2 * chunk + 64) + 63) / 64 * 64); }

// The passes of a top-k over n rows.  wide: the 512-query kernel; shadow: its
// scan of a q4 matrix's int8 shadow; wgs: workgroups that fill the chip.
// Every pass but the last ends on a whole chunk, so every workgroup's range
// starts at a multiple of the chunk (32, 64 or 128 rows).
inline std::vector<MqPass> mq_topk_passes(int64_t n, int64_t k, int chunk, int groups, int wgs, bool wide,
                                          bool shadow) {
    std::vector<MqPass> passes;
    auto whole = [&](int64_t rows) { return std::min<int64_t>(n, (rows + chunk - 1) / chunk * chunk); };
    // pass 0: everything is kept, so a workgroup takes at most rc - 2*chunk rows
    int64_t s = whole(std::max<int64_t>(8 * k, 4096));
    passes.push_back(mq_pass(0, s, chunk, groups, mq_region_keys(k, chunk) - 2 * chunk, wgs));
    if (s >= n) return passes;
    // later passes grow the prefix by g: about k*g keys per query reach
    // the select.  Fewest passes the select's buffer allows, then the
    // smallest g that still needs no more of them.
    const double span = (double)n / (double)s;
    const double gmax = std::max(4.0, (double)kMqSelectKeys / (double)k);
    int npass = std::max(1, (int)std::ceil(std::log(span) / std::log(gmax) - 1e-9));
    // the 512-query kernel appends about k*(g-1) pairs per query and
    // pass, each an exact test and an LDS atomic in the scan: keep g
    // near 4.5 (measured on 1024 queries over 1024x the first pass's
    // rows: 5 passes beat 3 by 4% of the step, 6 and 7 lose to 5 on the
    // selects)
    if (wide && !shadow) npass = std::max(npass, (int)std::ceil(std::log(span) / std::log(4.5) - 1e-9));
    // shadow pairs: every pair the select keeps is rescored from a random
    // row, so fewer, larger passes win as long as a pass's pairs (about
    // 4*k*g with the margins) fit the 512-thread select's 8K-key buffer,
    // which is what lets it prune before rescoring
    if (shadow) {
        const double gs = std::max(4.0, (8192.0 - (double)k) / (4.0 * (double)k));
        npass = std::max(1, (int)std::ceil(std::log(span) / std::log(gs) - 1e-9));
    }
    double g = std::pow(span, 1.0 / npass);
    // ... except its first growth pass, which grows the prefix by 16: over
    // so few rows the extra appends cost less than a pass and a select of
    // their own (1024 queries over 4M rows: 4,096 rows, then x16 and
    // three times x4 -- five passes instead of six -- measured 1,422 ->
    // 1,400 us a call; x8 gained nothing, x64 lost 35 us)
    double g0 = g;
    const double gfirst = std::min(16.0, gmax);
    if (wide && !shadow && span > gfirst * 4.5) {
        const double rest = span / gfirst;
        npass = 1 + (int)std::ceil(std::log(rest) / std::log(4.5) - 1e-9);
        g0 = gfirst;
        g = std::pow(rest, 1.0 / (npass - 1));
    }
    for (int i = 0; i < npass; i++) {
        const double gi = i == 0 ? g0 : g;
        const int64_t e = i + 1 == npass ? n : whole((int64_t)std::ceil(s * gi));
        if (e <= s) continue;
        passes.push_back(mq_pass(s, e, chunk, groups, 0, wgs));
        passes.back().grow = gi;
        s = e;
    }
    return passes;
}

}  // namespace manta
