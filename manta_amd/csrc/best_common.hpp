// best_common.hpp -- the k best of a workgroup's keys and of a query's parts
// for k <= kBestMaxK, by a floor and ranks instead of a streaming reservoir:
// shared by the score-row top-k (kernels_topk.hip) and the streaming scans
// (kernels_score.hip).
#pragma once

#include "device_common.hpp"
#include "kernels.hpp"
#include "mq_common.hpp"

namespace manta {

constexpr int kBestKeys = 1024;  // LDS keys of BestShared

struct BestShared {
    alignas(16) uint64_t keys[kBestKeys];
    TopKShared st;
    uint32_t floor;
    int cnt;
    int last;
};

// Keys above `mine` among keys[0..n) (n a multiple of 2; every lane reads the
// same address: LDS broadcasts, no dependent steps).
__device__ __forceinline__ int rank_in(const uint64_t* keys, int n, uint64_t mine) {
    int rank = 0;
#pragma unroll 16
    for (int i = 0; i < n; i += 2) {
        const ulonglong2 u = *(const ulonglong2*)(keys + i);
        rank += (u.x > mine ? 1 : 0) + (u.y > mine ? 1 : 0);
    }
    return rank;
}

// B.floor = the largest value with its low 12 bits clear that at least k of
// tops[0..64*N) reach (0 if fewer than k are above 0), by wave 0: one bit at a
// time, the lanes' comparisons counted by ballots.  20 steps of about 4 N
// instructions on one wave, where every thread ranking its own value among
// 256 took 1,000 on each (64 rows of 200,000, k = 100: 49 -> 26 us).
template <int N>
__device__ __forceinline__ void find_floor(const uint32_t* tops, int k, BestShared& B) {
    if (threadIdx.x >= 64) return;
    uint32_t t[N];
#pragma unroll
    for (int i = 0; i < N; i++) t[i] = tops[threadIdx.x + 64 * i];
    uint32_t floor = 0;
    for (uint32_t bit = 0x80000000u; bit >= 0x1000u; bit >>= 1) {
        const uint32_t cand = floor | bit;
        int reach = 0;
#pragma unroll
        for (int i = 0; i < N; i++) reach += __popcll(__ballot(t[i] >= cand));
        if (reach >= k) floor = cand;
    }
    if (threadIdx.x == 0) B.floor = floor;
}

// The `total` <= kBestKeys distinct keys in B.keys (whole workgroup of 256,
// after a barrier): the best min(k, total), sorted, to the front.
__device__ __forceinline__ int best_of(int total, int k, BestShared& B) {
    const int tid = threadIdx.x;
    if (total <= 256) {
        const uint64_t key = tid < total ? B.keys[tid] : 0ull;
        __syncthreads();
        if (tid >= total) B.keys[tid] = 0ull;  // rank_in reads pairs
        __syncthreads();
        const int rank = rank_in(B.keys, (total + 1) & ~1, key);
        __syncthreads();
        if (tid < total && rank < k) B.keys[rank] = key;
        __syncthreads();
        return total < k ? total : k;
    }
    if (tid == 0) B.st.cnt = total;
    __syncthreads();
    topk_compact(B.keys, &B.st, k);
    const int kept = B.st.cnt;
    topk_sort(B.keys, kept);
    return kept;
}

// The best min(k, held) of n keys offered in any order (keys at or above tau
// only), through the reservoir: key(i) for i in [0, n).
template <class A>
__device__ __forceinline__ int best_streamed(A key, int64_t n, uint64_t tau, int k, BestShared& B) {
    topk_init(B.keys, &B.st);
    for (int64_t base = 0; base < n; base += 256) {
        const int64_t i = base + threadIdx.x;
        const uint64_t t = B.st.tau > tau - 1 ? B.st.tau : tau - 1;
        topk_offer(i < n ? key(i) : 0ull, t, B.keys, &B.st);
        __syncthreads();
        topk_maybe_compact(B.keys, &B.st, k, kBestKeys);
    }
    topk_compact(B.keys, &B.st, k);
    const int kept = B.st.cnt;
    topk_sort(B.keys, kept);
    return kept;
}

// The best min(k, held) of the workgroup's scores, sorted, to B.keys as keys
// (k <= kBestMaxK; 256 threads, `count` scores each, or V when V > 0): order(j)
// is the order word of the thread's j-th, row(j) its index or -1 for none
// (whose order word is 0).  The k-th largest of the 256 threads' own best
// scores is a floor of the k-th (k distinct scores reach it), and few others
// do: 126 of 8,192 evenly spread ones for k = 100.  Those take their place by
// rank, with no round of histograms and no sort.  Returns how many keys there
// are, or -1 if more than kBestKeys reach the floor (scores arranged to, or
// many equal; the caller then streams them).
template <int V, class O, class R>
__device__ __forceinline__ int block_best(O order, R row, int count, int k, BestShared& B) {
    const int tid = threadIdx.x;
    const int n = V > 0 ? V : count;
    constexpr int U = V > 0 ? V : 4;
    uint32_t best = 0;
#pragma unroll U
    for (int j = 0; j < n; j++) {
        const uint32_t o = order(j);
        best = o > best ? o : best;
    }
    uint32_t* tops = (uint32_t*)B.keys;
    tops[tid] = best;
    if (tid == 0) B.cnt = 0;
    __syncthreads();
    find_floor<4>(tops, k, B);
    __syncthreads();
    const uint32_t floor = B.floor;
    int mine = 0;
    if (floor) {
#pragma unroll U
        for (int j = 0; j < n; j++) mine += order(j) >= floor ? 1 : 0;
    } else {
        for (int j = 0; j < n; j++) mine += row(j) >= 0 ? 1 : 0;
    }
    int pos = wave_append(mine, &B.cnt);
    __syncthreads();
    const int total = B.cnt;
    if (total > kBestKeys) return -1;
    if (mine) {
#pragma unroll U
        for (int j = 0; j < n; j++) {
            const uint32_t o = order(j);
            if (o >= floor && row(j) >= 0) B.keys[pos++] = ((uint64_t)o << 32) | (uint64_t)(~(uint32_t)row(j));
        }
    }
    __syncthreads();
    return best_of(total, k, B);
}

// End of a workgroup whose kept best keys (sorted) are in B.keys: publish
// them as part blockIdx.x of query qi; the last workgroup of the query
// (ticket) merges the gridDim.x <= kBestMaxParts parts into B.keys and resets
// the ticket.  Returns the merged count, or -1 in the workgroups that are not
// the last.  Publication as in finish_topk: agent-scope part stores, retired
// before the ticket.
//
// The parts are sorted, so the merge reads little of them: each is split into
// G lists by rank modulo G, 256 to 511 lists in all, whose heads are its
// first G keys; the k-th largest head is a floor, and each list is read only
// while it stays at or above it.
__device__ __forceinline__ int merge_best_parts(uint64_t* partial, uint32_t* tickets, int qi, int kept, int k,
                                                BestShared& B) {
    const int tid = threadIdx.x, P = (int)gridDim.x;
    uint64_t* part = partial + (int64_t)qi * P * k;
    uint64_t* dst = part + (int64_t)blockIdx.x * k;
    for (int i = tid; i < k; i += 256)
        __hip_atomic_store(dst + i, i < kept ? B.keys[i] : 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0)
        B.last = __hip_atomic_fetch_add(&tickets[qi], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                 (uint32_t)(P - 1);
    __syncthreads();
    if (!B.last) return -1;
    auto at = [&](int64_t i) {
        return (uint64_t)__hip_atomic_load(part + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    const int G = P >= 256 ? 1 : (255 + P) / P;
    const int lists = P * G;  // <= 512
    uint64_t head[2];
    uint32_t* tops = (uint32_t*)B.keys;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int l = tid + 256 * u, p = l / G, g = l - p * G;
        head[u] = l < lists && g < k ? at((int64_t)p * k + g) : 0ull;
    }
    tops[tid] = (uint32_t)(head[0] >> 32);
    tops[tid + 256] = (uint32_t)(head[1] >> 32);
    if (tid == 0) {
        B.cnt = 0;
        __hip_atomic_store(&tickets[qi], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    find_floor<8>(tops, k, B);
    __syncthreads();
    const uint64_t tau = ((uint64_t)B.floor << 32) | 1ull;  // (a key's low half is never 0)
#pragma unroll
    for (int u = 0; u < 2; u++) {
        if (head[u] < tau) continue;
        const int l = tid + 256 * u, p = l / G, g = l - p * G;
        uint64_t key = head[u];
        for (int r = g;;) {
            const int pos = atomicAdd(&B.cnt, 1);
            if (pos < kBestKeys) B.keys[pos] = key;
            r += G;
            if (r >= k) break;
            key = at((int64_t)p * k + r);
            if (key < tau) break;
        }
    }
    __syncthreads();
    const int total = B.cnt;
    if (total > kBestKeys) return best_streamed(at, (int64_t)P * k, tau, k, B);
    return best_of(total, k, B);
}

}  // namespace manta
