// stream_plan.hpp -- launch shapes of the streaming scans (host arithmetic
// only: no HIP types, so that it also compiles by itself).
#pragma once

#include <stdint.h>

#include <algorithm>

namespace manta {

// Rounds of 256 rows per scan workgroup, for about `wgs` workgroups in all,
// so each streams a long contiguous range and the per-workgroup prologue and
// top-k publication are paid rarely.  The fused top-k takes one workgroup
// per CU (C0's 32 problems: 82.3 us a launch against 85.1 with two per CU,
// 97.6 with one per two CUs and 99.2 with 1.25 per CU); the score matrix
// keeps two per CU.
inline int choose_rounds(int64_t tiles, int64_t nq, int64_t wgs) {
    int64_t r = (tiles * nq + wgs - 1) / wgs;
    // small calls are latency-bound: two rounds halve the parts the last
    // workgroup merges (one 65536 x 256 query, with the lists filled and
    // merged by rank: 13.3 us a call against 15.8 with one round and 14.1
    // with four)
    if (r < 2 && tiles >= 4) r = 2;
    // never more rounds than the rows have tiles (many queries over few rows):
    // the workgroup would run them, and hold LDS for them, on no rows
    return (int)std::max<int64_t>(1, std::min<int64_t>({64, r, tiles}));
}

// Rounds of a selection that buffers its scores, `pitch` bytes a row.  A
// workgroup holds a KB of LDS a round (and up to 80 KB beside them), so at the
// rounds that spread the rows over one workgroup per CU a CU may take no
// second one, and the few workgroups past a whole wave cost another: 43 parts
// for each of 6 queries are 258 on 256 CUs.  Parts that make one or two whole
// waves, where those are not too long for the row's width; else short parts,
// many a CU.  Before and now, us, q4 dot, k = 5: 6 x 700,000 x 384 321 and 163,
// 7 x 700,000 x 384 330 and 146, 7 x 1,200,000 x 384 485 and 322.
inline int buffered_rounds(int64_t tiles, int64_t nq, int64_t wgs, int rounds, int64_t max_parts, int pitch) {
    if (nq * ((tiles + rounds - 1) / rounds) <= wgs) return rounds;
    for (int waves = 1; waves <= 2; waves++) {
        const int64_t parts = std::min(tiles, wgs * waves / nq);
        if (parts < 1 || parts > max_parts) continue;
        const int64_t r = (tiles + parts - 1) / parts;
        // (narrow rows want more wavefronts in flight than one workgroup's;
        // wide ones keep the memory busy with it)
        if (r <= (waves == 1 ? (pitch >= 128 ? 64 : 0) : (pitch >= 320 ? 64 : 40))) return (int)r;
    }
    return (int)std::min<int64_t>(rounds, std::max<int64_t>(24, (tiles + max_parts - 1) / max_parts));
}

// Little work: the multi-query passes' launches (encoding, then a scan and a
// select each) would cost more than one streaming launch that reads the cached
// rows once per query.  The work of a row and query is its d values and a part
// (256 of them) that no width saves.  Whole reference calls, cosine, k = 10, us
// in passes / streaming, by nq x n x d:
//
//   inside       32 x 39,877 x 128 q8   55 / 36    32 x 17,889 x 600 q8   59 / 55
//                8 x 79,753 x 512 q4    64 / 54    32 x 12,191 x 1,000 q8 62 / 55
//   past it      32 x 39,063 x 384 q8   57 / 55    8 x 156,251 x 384 q8   62 / 99
//                32 x 32,553 x 512 q4   62 / 70    32 x 24,415 x 768 q8   65 / 65
//   one pass     128 x 3,397 x 480 q8   43 / 44    200 x 2,400 x 384 q8   43 / 47
//                512 x 1,200 x 256 q8   40 / 33    300 x 2,400 x 256 q4   74 / 42
//   ... wide     128 x 1,145 x 768 q8   37 / 35    200 x 1,200 x 768 q8   39 / 52
//                128 x 1,013 x 900 q8   40 / 35    128 x 2,289 x 768 q4   43 / 53
//
// Up to 4,096 rows the passes are one and cost two thirds of three (q4's a
// little more than q8's), so less work pays for them, least for wide rows.
// Where the sides differ little the line is not fitted: 8 x 59,815 x 768 q8
// still streams, 65 / 78.
inline bool stream_is_faster(bool q8, int64_t n, int64_t d, int64_t nq) {
    const bool one_pass = n <= 4096;
    double line = q8 && one_pass ? 3e8 : 5e8;
    if (one_pass && d > 512) line /= 2;
    return (double)nq * (double)n * (double)(d + 256) < line;
}

}  // namespace manta
