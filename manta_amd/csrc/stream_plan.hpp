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

// Little work: the multi-query passes' launches (encoding, then a scan and a
// select each) would cost more than one streaming launch that reads the cached
// rows once per query.  Whole reference calls, passes against streaming: q8, 8 queries x
// 80,000 x 384 67 / 57 us, 32 x 20,000 x 256 64 / 50; past the line 8 x 50,000 x
// 768 and 8 x 200,000 x 128 are even, 100 x 4,000 x 1,000 streams in 168 against
// 103.  Up to 4,096 q8 rows the passes are one, and 512 x 1,200 x 256 takes 52
// against 63.
inline bool stream_is_faster(bool q8, int64_t n, int64_t d, int64_t nq) {
    const double limit = q8 && n <= 4096 ? 3e8 : 5e8;
    return (double)nq * (double)n * (double)(d + 256) < limit;
}

}  // namespace manta
