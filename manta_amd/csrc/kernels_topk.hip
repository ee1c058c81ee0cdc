// kernels_topk.hip -- top-k selection (topKTensor, runtime/backend/
// tensor_ops.go:1523-1592) over f32 score rows, and the candidate pack.
//
// k <= 192 (topk_rows_kernel, one launch): grid (parts, rows); a workgroup
// holds a segment of one row in registers, finds its k best (block_best) and
// publishes them; the last workgroup of the row merges the parts the same
// way.  Larger k: topk_rows_partial_kernel streams a segment in rounds of 256
// scores through the LDS reservoir, topk_merge_kernel reduces a row's parts.
// Results are sorted by (value desc, index asc) -- or (value asc, index asc)
// for smallest-k.  Keys make the order total, so the result does not
// depend on how rows were split across workgroups.
#include "best_common.hpp"
#include "device_common.hpp"
#include "kernels.hpp"

namespace manta {

// One workgroup per segment of 256*V scores, one launch for the whole top-k:
// the last workgroup of a row (ticket) merges the parts.  Publication as in
// finish_topk: agent-scope part stores, retired before the ticket.  What
// bounds it is the read of the scores; the streaming reservoir (a barrier
// pair per 256 scores) and its merge launch took 62 + 27 us for 64 rows of
// 200,000 and k = 100, this kernel 26 us.
template <int V, bool VEC>
__global__ __launch_bounds__(256) void topk_rows_kernel(const float* __restrict__ scores, int64_t cols, int k,
                                                        int smallest, uint64_t* __restrict__ partial,
                                                        uint32_t* __restrict__ tickets, int32_t* __restrict__ ids,
                                                        float* __restrict__ values) {
    __shared__ BestShared B;
    const int tid = threadIdx.x;
    const int64_t row = blockIdx.y;
    const int P = (int)gridDim.x;
    const float* src = scores + row * cols;
    const int64_t c0 = (int64_t)blockIdx.x * (256 * V);
    const int left = cols - c0 < 256 * V ? (int)(cols - c0) : 256 * V;
    // thread t's j-th score: four in a row at a time (VEC), else one
    auto at = [&](int j) { return VEC ? ((j >> 2) * 256 + tid) * 4 + (j & 3) : j * 256 + tid; };
    uint32_t o[V];
#pragma unroll
    for (int j = 0; j < V; j += VEC ? 4 : 1) {
        const int c = at(j);
        if (VEC) {
            // (cols % 4 == 0: the four are all inside or all outside)
            const float4 f = c < left ? *(const float4*)(src + c0 + c) : float4{0, 0, 0, 0};
            o[j] = __float_as_uint(f.x), o[j + 1] = __float_as_uint(f.y);
            o[j + 2] = __float_as_uint(f.z), o[j + 3] = __float_as_uint(f.w);
        } else {
            o[j] = __float_as_uint(c < left ? src[c0 + c] : 0.0f);
        }
    }
#pragma unroll
    for (int j = 0; j < V; j++) {
        o[j] = float_order(__uint_as_float(o[j]));
        if (smallest) o[j] = ~o[j];
    }
    if (left < 256 * V) {
#pragma unroll
        for (int j = 0; j < V; j++) o[j] = at(j) < left ? o[j] : 0u;
    }
    int kept = block_best<V>([&](int j) { return o[j]; },
                             [&](int j) { return at(j) < left ? (int)(c0 + at(j)) : -1; }, V, k, B);
    if (kept < 0)
        kept = best_streamed([&](int64_t i) { return make_key(src[c0 + i], (uint32_t)(c0 + i), smallest); }, left,
                             1ull, k, B);
    if (P > 1) {
        kept = merge_best_parts(partial, tickets, (int)row, kept, k, B);
        if (kept < 0) return;
    }
    for (int i = tid; i < k; i += 256) {
        const uint64_t key = i < kept ? B.keys[i] : 0ull;
        ids[row * k + i] = key ? (int32_t)key_index(key) : -1;
        if (values) values[row * k + i] = key ? key_score(key, smallest) : 0.0f;
    }
}

// Scores a thread holds: 16 while that leaves few workgroups (one part per
// 4,096 scores; latency), else 32, else 64; 0 when the parts would be too many
// for the merge or k is too large (the two-launch path).
static int topk_rows_v(int64_t rows, int64_t cols, int64_t k) {
    if (k > kBestMaxK) return 0;
    auto parts = [&](int v) { return (cols + 256 * v - 1) / (256 * v); };
    for (int v = 16; v <= 64; v <<= 1)
        if ((v == 64 || rows * parts(v) <= 2048 || parts(2 * v) == parts(v)) && parts(v) <= kBestMaxParts) return v;
    return 0;
}

int64_t topk_rows_parts(int64_t rows, int64_t cols, int64_t k) {
    const int v = topk_rows_v(rows, cols, k);
    return v ? (cols + 256 * v - 1) / (256 * v) : 0;
}

hipError_t launch_topk_rows(const float* scores, int64_t rows, int64_t cols, int k, int smallest, uint64_t* partial,
                            uint32_t* tickets, int32_t* ids, float* values, hipStream_t s) {
    const int v = topk_rows_v(rows, cols, k);
    if (!v || rows <= 0 || rows > 65535 || k <= 0 || k > cols) return hipErrorInvalidValue;
    const dim3 grid((unsigned)topk_rows_parts(rows, cols, k), (unsigned)rows);
    const bool vec = cols % 4 == 0 && ((uintptr_t)scores & 15) == 0;
#define MANTA_TOPK(V, VEC) \
    hipLaunchKernelGGL((topk_rows_kernel<V, VEC>), grid, dim3(256), 0, s, scores, cols, k, smallest, partial, \
                       tickets, ids, values)
    if (v == 16) { if (vec) MANTA_TOPK(16, true); else MANTA_TOPK(16, false); }
    else if (v == 32) { if (vec) MANTA_TOPK(32, true); else MANTA_TOPK(32, false); }
    else { if (vec) MANTA_TOPK(64, true); else MANTA_TOPK(64, false); }
#undef MANTA_TOPK
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void topk_rows_partial_kernel(const float* __restrict__ scores,
                                                                int64_t cols, int64_t seg, int k,
                                                                int cap, int smallest,
                                                                uint64_t* __restrict__ partial) {
    extern __shared__ uint64_t keys[];
    __shared__ TopKShared st;
    const int64_t row = blockIdx.y;
    const float* src = scores + row * cols;
    const int64_t c0 = (int64_t)blockIdx.x * seg;
    int64_t c1 = c0 + seg;
    if (c1 > cols) c1 = cols;
    topk_init(keys, &st);
    for (int64_t base = c0; base < c1; base += blockDim.x) {
        const int64_t c = base + threadIdx.x;
        uint64_t key = 0;
        if (c < c1) key = make_key(src[c], (uint32_t)c, smallest);
        topk_offer(key, st.tau, keys, &st);
        __syncthreads();
        topk_maybe_compact(keys, &st, k, cap);
    }
    topk_compact(keys, &st, k);
    uint64_t* dst = partial + (row * gridDim.x + blockIdx.x) * k;
    for (int i = threadIdx.x; i < k; i += blockDim.x) dst[i] = i < st.cnt ? keys[i] : 0ull;
}

__global__ __launch_bounds__(256) void topk_merge_kernel(const uint64_t* __restrict__ partial,
                                                         int64_t per_row, int k, int cap,
                                                         int smallest, int32_t* __restrict__ ids,
                                                         float* __restrict__ values) {
    extern __shared__ uint64_t keys[];
    __shared__ TopKShared st;
    const int64_t row = blockIdx.x;
    const uint64_t* src = partial + row * per_row;
    topk_init(keys, &st);
    for (int64_t base = 0; base < per_row; base += blockDim.x) {
        const int64_t i = base + threadIdx.x;
        uint64_t key = i < per_row ? src[i] : 0ull;
        topk_offer(key, st.tau, keys, &st);
        __syncthreads();
        topk_maybe_compact(keys, &st, k, cap);
    }
    topk_compact(keys, &st, k);
    const int kept = st.cnt;
    topk_sort(keys, kept);
    for (int i = threadIdx.x; i < k; i += blockDim.x) {
        uint64_t key = i < kept ? keys[i] : 0ull;
        ids[row * k + i] = key ? (int32_t)key_index(key) : -1;
        if (values) values[row * k + i] = key ? key_score(key, smallest) : 0.0f;
    }
}

hipError_t launch_topk_rows_partial(const float* scores, int64_t rows, int64_t cols, int64_t seg,
                                    int parts, int k, int cap, int smallest, uint64_t* partial,
                                    hipStream_t s) {
    hipLaunchKernelGGL(topk_rows_partial_kernel, dim3(parts, (unsigned)rows), dim3(256),
                       (size_t)cap * sizeof(uint64_t), s, scores, cols, seg, k, cap, smallest,
                       partial);
    return hipGetLastError();
}

hipError_t launch_topk_merge(const uint64_t* partial, int64_t rows, int64_t per_row, int k, int cap,
                             int smallest, int32_t* ids, float* values, hipStream_t s) {
    hipLaunchKernelGGL(topk_merge_kernel, dim3((unsigned)rows), dim3(256),
                       (size_t)cap * sizeof(uint64_t), s, partial, per_row, k, cap, smallest, ids,
                       values);
    return hipGetLastError();
}

// ------------------------------------------------------ candidate pack

// One wave per (query, rank): the candidate id (int64), the packed row's
// bytes (4-byte words when row_bytes and pitch allow, else bytes) and its
// scales.  An index outside [0, n) zero-fills the slot and is reported.
__global__ __launch_bounds__(256) void pack_candidates_kernel(PackArgs a) {
    const int64_t slot = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (slot >= a.nq * a.k) return;
    const int lane = threadIdx.x & 63;
    const int64_t q = slot / a.k;
    const int idx = a.top[slot];
    const bool ok = idx >= 0 && (int64_t)idx < a.n;
    if (!ok && lane == 0) report_gather_error(a.err, slot, idx);
    const int64_t row = (a.sets == 1 ? 0 : q * a.n) + (ok ? idx : 0);
    if (a.ids_out && lane == 0) a.ids_out[slot] = (a.ids && ok) ? a.ids[row] : 0;
    uint8_t* dst = a.rows_out + slot * a.row_bytes;
    const uint8_t* src = a.codes + row * a.pitch;
    if ((a.row_bytes & 3) == 0 && (a.pitch & 3) == 0) {
        for (int w = lane; w < a.row_bytes / 4; w += 64)
            ((uint32_t*)dst)[w] = ok ? ((const uint32_t*)src)[w] : 0u;
    } else {
        for (int b = lane; b < a.row_bytes; b += 64) dst[b] = ok ? src[b] : (uint8_t)0;
    }
    uint8_t* sdst = a.scales_out + slot * a.scale_bytes;
    const uint8_t* ssrc = a.scales + row * a.scale_bytes;
    for (int b = lane; b < a.scale_bytes; b += 64) sdst[b] = ok ? ssrc[b] : (uint8_t)0;
}

hipError_t launch_pack_candidates(const PackArgs& a, hipStream_t s) {
    const int64_t slots = a.nq * a.k;
    hipLaunchKernelGGL(pack_candidates_kernel, dim3((unsigned)((slots + 3) / 4)), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace manta
