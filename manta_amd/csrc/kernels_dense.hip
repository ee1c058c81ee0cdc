// kernels_dense.hip -- scores of f32 query vectors against dense f32 / f16
// retrieval vectors with the reference's arithmetic: dotRetrievalVectors
// (runtime/retrieval_eval.go:651-661), `sum += a[i]*b[i]` in f32 over
// i < min(len(a), len(b)), every product and sum rounded on its own (no
// FMA), in index order.
//
// The order of operations is fixed, so the work cannot be reassociated onto
// the matrix cores: each (query, row) pair is one sequential chain of
// v_mul_f32 + v_add_f32, and what bounds many queries is those two
// instructions per element and pair: 9.8 G lane instructions for 64 f32 queries
// against 200,000 x 384 rows, 170 us at the 58 T/s that a loop of nothing but
// such pairs reaches on this card (63 us to copy the rows).
//
// Tiles: a workgroup takes RT rows x QT queries, KC elements of each at a
// time staged through LDS transposed ([element][row], [element][query]); a
// thread owns TR rows x TQ queries, so an element's TR + TQ LDS values feed
// 2*TR*TQ VALU instructions.  The next KC elements are in registers while the
// current ones are summed.  Rows of f16 values are widened exactly.  Elements
// past the common length are staged as zeros on both sides: a partial sum is
// never -0 (it starts at +0), so adding 0 * 0 leaves it as it is.  A lane
// reading its own row's 16 bytes at a time (1536 bytes apart), every row again
// for each 8 queries, took 2,506 us on that shape; these tiles 242-255 us
// (the LDS reads, TR + TQ values for 2*TR*TQ instructions, and the staging
// issue beside them).
// Output: the f32 score matrix [nq][n] (the top-k runs on it afterwards).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "device_common.hpp"
#include "kernels.hpp"

#pragma clang fp contract(off)

namespace manta {

namespace {

constexpr int kDenseKC = 32;  // elements staged at a time

template <typename T>
__device__ __forceinline__ float widen(T x);
template <>
__device__ __forceinline__ float widen<float>(float x) {
    return x;
}
template <>
__device__ __forceinline__ float widen<uint16_t>(uint16_t x) {
    return h2f(x);
}

// VEC: rows are 16-byte aligned and hold whole 16-byte groups of the first
// `len` elements (len * sizeof(T) % 16 == 0 and the row pitch likewise).
// 256 threads: QG groups of TQ queries x 256/QG groups of TR rows.
template <typename T, bool VEC, int QG, int TQ, int TR>
__global__ __launch_bounds__(256) void dense_dot_kernel(const T* __restrict__ rows, int64_t n, int64_t pitch,
                                                        int len, const float* __restrict__ queries, int64_t qpitch,
                                                        int nq, int qtiles, float* __restrict__ out) {
    constexpr int KC = kDenseKC;
    constexpr int QT = QG * TQ, RG = 256 / QG, RT = RG * TR;
    constexpr int W = VEC ? 16 / (int)sizeof(T) : 1;  // elements per load
    constexpr int LPR = KC / W;                       // lanes per row and stage
    constexpr int RPP = 256 / LPR;                    // rows per pass of the workgroup
    constexpr int NP = RT / RPP;
    constexpr int NQ = (QT * KC + 255) / 256;
    static_assert(RT % RPP == 0, "passes tile the rows");
    __shared__ float As[KC][RT + 4];
    __shared__ float Bs[KC][QT + 4];
    const int tid = threadIdx.x;
    const int64_t rt = blockIdx.x / (unsigned)qtiles;
    const int q0 = (int)(blockIdx.x - rt * qtiles) * QT;
    const int64_t r0 = rt * RT;
    const int lr = tid / LPR, lc = (tid % LPR) * W;

    T ra[NP][W];
    float rq[NQ];
    auto load = [&](int k0) {
        const int c = k0 + lc;
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const int64_t row = r0 + p * RPP + lr;
            const bool in = row < n && c < len;
            const T* src = rows + row * pitch + c;
            if (VEC) {
                *(uint4*)ra[p] = in ? *(const uint4*)src : uint4{0, 0, 0, 0};
            } else {
                ra[p][0] = in ? *src : (T)0;
            }
        }
#pragma unroll
        for (int i = 0; i < NQ; i++) {
            const int e = tid + 256 * i, q = e / KC, kk = e % KC;
            const bool in = q < QT && q0 + q < nq && k0 + kk < len;
            rq[i] = in ? queries[(int64_t)(q0 + q) * qpitch + k0 + kk] : 0.0f;
        }
    };
    auto stage = [&]() {
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int e = 0; e < W; e++) As[lc + e][p * RPP + lr] = widen<T>(ra[p][e]);
#pragma unroll
        for (int i = 0; i < NQ; i++) {
            const int e = tid + 256 * i, q = e / KC, kk = e % KC;
            if (q < QT) Bs[kk][q] = rq[i];
        }
    };

    const int qg = tid % QG, rg = tid / QG;
    float acc[TQ][TR];
#pragma unroll
    for (int j = 0; j < TQ; j++)
#pragma unroll
        for (int i = 0; i < TR; i++) acc[j][i] = 0.0f;
    load(0);
    for (int k0 = 0; k0 < len; k0 += KC) {
        stage();
        __syncthreads();
        if (k0 + KC < len) load(k0 + KC);
#pragma unroll 8
        for (int kk = 0; kk < KC; kk++) {
            float x[TR], y[TQ];
#pragma unroll
            for (int i = 0; i < TR; i++) x[i] = As[kk][rg * TR + i];
            // (a query group's TQ values lie 4 at a time, QG groups side by
            // side, so the lanes of a wave read consecutive 16-byte pieces)
#pragma unroll
            for (int j = 0; j < TQ; j++) y[j] = Bs[kk][(j / 4) * 4 * QG + qg * 4 + j % 4];
#pragma unroll
            for (int j = 0; j < TQ; j++)
#pragma unroll
                for (int i = 0; i < TR; i++) acc[j][i] = fadd_rn(acc[j][i], fmul_rn(y[j], x[i]));
        }
        __syncthreads();
    }
    const int64_t row = r0 + rg * TR;
#pragma unroll
    for (int j = 0; j < TQ; j++) {
        const int q = q0 + (j / 4) * 4 * QG + qg * 4 + j % 4;
        if (q >= nq) continue;
#pragma unroll
        for (int i = 0; i < TR; i++)
            if (row + i < n) out[(int64_t)q * n + row + i] = acc[j][i];
    }
}

template <typename T, int QG, int TQ, int TR>
hipError_t launch_dense_tile(const T* rows, int64_t n, int64_t pitch, int len, const float* queries, int64_t qpitch,
                             int nq, float* out, hipStream_t s) {
    const int64_t rtiles = (n + 256 / QG * TR - 1) / (256 / QG * TR);
    const int qtiles = (nq + QG * TQ - 1) / (QG * TQ);
    if (rtiles * qtiles > 0x7FFFFFFF) return hipErrorInvalidValue;
    constexpr int W = 16 / sizeof(T);
    const bool vec = len % W == 0 && pitch % W == 0 && ((uintptr_t)rows & 15) == 0;
    const dim3 grid((unsigned)(rtiles * qtiles));
    if (vec) hipLaunchKernelGGL((dense_dot_kernel<T, true, QG, TQ, TR>), grid, dim3(256), 0, s, rows, n, pitch, len,
                                queries, qpitch, nq, qtiles, out);
    else hipLaunchKernelGGL((dense_dot_kernel<T, false, QG, TQ, TR>), grid, dim3(256), 0, s, rows, n, pitch, len,
                            queries, qpitch, nq, qtiles, out);
    return hipGetLastError();
}

// Queries per tile: the smallest that takes all queries at once, up to 64
// (fewer re-reads of the rows), halved while the grid leaves CUs idle.
template <typename T>
hipError_t launch_dense_dot_t(const T* rows, int64_t n, int64_t pitch, int len, const float* queries,
                              int64_t qpitch, int nq, float* out, hipStream_t s) {
    int qt = 4;
    while (qt < 64 && qt < nq) qt <<= 1;
    auto groups = [&](int q) { return ((n + (q == 64 ? 127 : 255)) / (q == 64 ? 128 : 256)) * ((nq + q - 1) / q); };
    while (qt > 4 && groups(qt) < 256) qt >>= 1;
#define MANTA_DENSE(QG, TQ, TR) launch_dense_tile<T, QG, TQ, TR>(rows, n, pitch, len, queries, qpitch, nq, out, s)
    switch (qt) {
        case 64: return MANTA_DENSE(8, 8, 4);
        case 32: return MANTA_DENSE(4, 8, 4);
        case 16: return MANTA_DENSE(2, 8, 2);
        case 8: return MANTA_DENSE(1, 8, 1);
        default: return MANTA_DENSE(1, 4, 1);
    }
#undef MANTA_DENSE
}

}  // namespace

hipError_t launch_dense_dot(const void* rows, int f16, int64_t n, int64_t pitch, int len, const float* queries,
                            int64_t qpitch, int nq, float* out, hipStream_t s) {
    if (n <= 0 || nq <= 0 || len < 0) return hipErrorInvalidValue;
    return f16 ? launch_dense_dot_t<uint16_t>((const uint16_t*)rows, n, pitch, len, queries, qpitch, nq, out, s)
               : launch_dense_dot_t<float>((const float*)rows, n, pitch, len, queries, qpitch, nq, out, s);
}

}  // namespace manta
