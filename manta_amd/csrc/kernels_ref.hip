// kernels_ref.hip -- scores with the reference's own arithmetic (dotRows,
// cosineRows, l2DistanceRows; runtime/backend/tensor_ops.go:1366-1490) on the
// values packed q8 / q4 rows stand for.
//
// ref_rescore_kernel (16 lanes a row; ref_rescore_rows_kernel, a row a thread,
// for many): the quantized-query scans return their best kp rows; each is
// rescored with the reference arithmetic.
// ref_finish_kernel (one workgroup per query) sorts them by (score, index)
// as topKTensor does
// (tensor_ops.go:1539-1551), and keeps the best k if the bounds of
// ref_common.hpp prove that no row outside the kp can reach the k-th: for
// largest-first, every outside row has a scan score of at most that of the
// kp-th row, c, hence a reference score of at most ref_hi(c), and the proof
// is ref_hi(c) < L with L the k-th best reference score found (smallest-
// first: ref_lo(c) > L).  Otherwise the query is marked for ref_scan.
//
// ref_scores_kernel: the score matrix, each pair its own sequential chain.
// ref_scan_kernel: lane = row, the reference score of every row; writes the
// score matrix (q4, one or two queries), or feeds the streaming reservoir (device_common.hpp) and the
// last-workgroup merge (scan_common.hpp) for the queries marked by the
// finish, from the threshold key L gives.
#include "device_common.hpp"
#include "kernels.hpp"
#include "mq_common.hpp"
#include "ref_common.hpp"
#include "scan_common.hpp"

namespace manta {

template <int FMT, int OP>
__device__ __forceinline__ float ref_row_score(const void* codes, const void* scales, const double* sqd,
                                               int64_t row, int pitch, int d, const float* qf, double sqn) {
    const double dn = OP == OP_COSINE ? sqd[row] : 0.0;
    if (FMT == 8)
        return ref_score_q8<OP>(qf, (const int8_t*)codes + row * pitch, ((const float*)scales)[row], d, sqn, dn);
    return ref_score_q4<OP>(qf, (const uint8_t*)codes + row * pitch, (const uint16_t*)scales + row * (d / 32), d,
                            sqn, dn);
}

// Floats of an LDS row of d values: 4 past a multiple of 64, so that rows
// read side by side start on different banks.
__host__ __device__ constexpr int ref_row_pitch(int d) { return (d + 63) / 64 * 64 + 4; }

// Keys of the finish: next_pow2(kp) <= kRefMaxKeys in LDS.
constexpr int kRefMaxKeys = 4096;

// ------------------------------------------------ 16 lanes a row

// Values a lane of 16 holds: 8 bytes of codes in turn, q8 pieces of 8 columns,
// q4 pieces of 16 (half a block); up to 8 (q8) or 4 (q4) pieces for d <= 1024.
template <int FMT>
struct RefPiece {
    static constexpr int COLS = FMT == 8 ? 8 : 16, MAX = kMaxQueryDim / (16 * COLS);
};

template <int CTRL>
__device__ __forceinline__ double dpp_dbl(double x) {
    const uint64_t b = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, false);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
// Sum over each 16-lane row (quad xor 1, xor 2, half mirror, mirror).
__device__ __forceinline__ double row16_dsum(double s) {
    s += dpp_dbl<0xB1>(s);
    s += dpp_dbl<0x4E>(s);
    s += dpp_dbl<0x141>(s);
    return s + dpp_dbl<0x140>(s);
}

// A query's f16 elements are integers times 2^(t - 24), t the fewest trailing
// zeros among them, so the squares are multiples of 2^(2t - 48): while their
// sum stays below 2^(2t + 5) every partial sum in any order is exact, and one
// taken in any order is the reference's sequential one.  (Infinities and NaN:
// not below.)
__device__ __forceinline__ bool norm_exact(double sum, int t) {
    return sum < __builtin_ldexp(1.0, 2 * (t < 40 ? t : 0) + 5);
}

// sqrt of the query's f64 square-sum by 16 lanes (lane 0 gets it).
__device__ __forceinline__ double ref_norm16(const float* qf, int d) {
    const int i16 = threadIdx.x & 15;
    double s = 0.0;
    int t = 64;
    for (int c = i16; c < d; c += 16) {
        const double x = (double)qf[c];
        s = __fma_rn(x, x, s);
        // (an f16 value in f32: 24-bit significand, exponent bits e - 127)
        const uint32_t b = __builtin_bit_cast(uint32_t, qf[c]);
        const int tc = __builtin_ctz((b & 0x7fffffu) | 0x800000u) + (int)((b >> 23) & 255) - (127 + 23 - 24);
        if ((b << 1) != 0 && tc < t) t = tc;
    }
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
        const int o = __shfl_xor(t, off);
        t = o < t ? o : t;
    }
    s = row16_dsum(s);
    if (i16 != 0) return 0.0;
    return norm_exact(s, t) ? sqrt_rn(s) : ref_sqrt_norm(qf, d);
}

// The reference score from a sum s of its f64 terms taken in another order, if
// that order cannot matter: the sequential sum differs from s by at most err
// (both rounding errors together), the end of the arithmetic is monotone in
// the sum (its own f64 roundings widen the ends by 2^-50), and both ends narrow
// to the same float.  NaN: not decided.
template <int OP>
__device__ __forceinline__ bool ref_narrow(double s, double err, double den, float& out) {
    double lo = s - err, hi = s + err;
    const double w = 8.8817841970012523e-16;  // 2^-50
    if (OP == OP_COSINE) {
        if (den == 0.0) {
            out = 0.0f;
            return true;
        }
        lo = lo / den, hi = hi / den;
        lo -= __builtin_fabs(lo) * w;
        hi += __builtin_fabs(hi) * w;
    } else {
        lo = __builtin_sqrt(lo > 0.0 ? lo : 0.0) * (1.0 - w);
        hi = __builtin_sqrt(hi) * (1.0 + w);
    }
    out = (float)lo;
    // (bit patterns: -0 and +0 are different results)
    return __float_as_uint((float)lo) == __float_as_uint((float)hi) && lo <= hi && lo > -3e38 && hi < 3e38;
}

// Reference keys of the scan's kp candidates of query blockIdx.y, 16 a
// workgroup and 16 lanes a row: keys [nq][kp] (0 for an invalid id).
// cosine / l2: the lanes' partial f64 sums are added across the row and
// ref_narrow decides; where it cannot (a few candidates in 10^5: theirs are the
// large scores, of coarse floats) the row goes through LDS and a lane runs the
// sequential sum.  dot: an
// f32 chain has no such slack, so the lanes only dequantize the rows into LDS
// and a lane per row runs the chain.  A candidate per thread ran every
// conversion and f64 step of its row, and one thread the query's norm, in one
// chain: 4 queries x 28 candidates of d = 384 took 18 us, now 6.3.
template <int FMT, int OP>
__global__ __launch_bounds__(256) void ref_rescore_kernel(RefArgs a, uint64_t* __restrict__ keys) {
    typedef RefPiece<FMT> RP;
    extern __shared__ __attribute__((aligned(16))) float smem[];
    __shared__ double norm_s[4];
    __shared__ int norm_t[4];
    const int tid = threadIdx.x, i16 = tid & 15, g = tid >> 4;
    const int d = a.d;
    const int P = ref_row_pitch(d);
    float* qf = smem;        // [P]
    float* vals = smem + P;  // [16][P] (dot: a row each), or [4][P] (a row a wave)
    const int q0 = (int)blockIdx.y;
    const int at = (int)blockIdx.x * 16 + g;
    const bool has = at < a.kp;
    const int32_t cid = has ? a.cand_ids[(int64_t)q0 * a.kp + at] : -1;
    const bool ok = cid >= 0 && (int64_t)cid < a.n;
    const int64_t row = (int64_t)q0 * a.set_stride + (ok ? cid : 0);
    // the row's pieces, all loads at once
    const uint8_t* src = (const uint8_t*)a.codes + row * a.pitch + 8 * i16;
    const int pieces = (d + RP::COLS - 1) / RP::COLS;
    uint2 w[RP::MAX];
    float sc[RP::MAX];
#pragma unroll
    for (int j = 0; j < RP::MAX; j++) {
        const int p = 16 * j + i16;
        w[j] = uint2{0, 0};
        sc[j] = 0.0f;
        if (p < pieces) {
            w[j] = *(const uint2*)(src + 128 * j);
            sc[j] = FMT == 8 ? ((const float*)a.scales)[row]
                             : h2f(((const uint16_t*)a.scales)[row * (d / 32) + (p >> 1)]);
        }
    }
    const double sqd = OP == OP_COSINE ? a.sqd[row] : 0.0;
    // the query, and with it the norm's sum (exact in any order, or run again in
    // column order: norm_exact)
    double nsum = 0.0;
    int nt = 64;
    for (int c = tid; c < d; c += 256) {
        const uint16_t h = a.queries[(int64_t)q0 * d + c];
        const float x = h2f(h);
        qf[c] = x;
        if (OP == OP_COSINE) {
            nsum = __fma_rn((double)x, (double)x, nsum);
            const int e = (h >> 10) & 31;
            const uint32_t m = (h & 0x3ffu) | (e ? 0x400u : 0u);
            const int t = m ? __builtin_ctz(m) + (e ? e - 1 : 0) : 64;
            nt = t < nt ? t : nt;
        }
    }
    if (OP == OP_COSINE) {
        nsum = row16_dsum(nsum);
        nsum += __shfl_xor(nsum, 16);
        nsum += __shfl_xor(nsum, 32);
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int o = __shfl_xor(nt, off);
            nt = o < nt ? o : nt;
        }
        if ((tid & 63) == 0) {
            norm_s[tid >> 6] = nsum;
            norm_t[tid >> 6] = nt;
        }
    }
    __syncthreads();
    double sqn = 0.0;
    if (OP == OP_COSINE) {
        nsum = (norm_s[0] + norm_s[1]) + (norm_s[2] + norm_s[3]);
        nt = norm_t[0];
        for (int i = 1; i < 4; i++) nt = norm_t[i] < nt ? norm_t[i] : nt;
        sqn = norm_exact(nsum, nt) ? sqrt_rn(nsum) : ref_sqrt_norm(qf, d);
    }
    auto value = [&](int j, int e) {
        const uint32_t word = FMT == 8 ? (e < 4 ? w[j].x : w[j].y) : (e < 8 ? w[j].x : w[j].y);
        const int code = FMT == 8 ? (int)(word << (24 - 8 * (e & 3))) >> 24 : (int)(word << (28 - 4 * (e & 7))) >> 28;
        return fmul_rn((float)code, sc[j]);
    };
    // a row's values to LDS by its 16 lanes; the sequential sum over them by one
    auto write_row = [&](float* v) {
#pragma unroll
        for (int j = 0; j < RP::MAX; j++) {
            // (opaque: or the sums' converted values are kept for here, 64 registers)
            asm volatile("" : "+v"(w[j].x), "+v"(w[j].y));
            const int c0 = (16 * j + i16) * RP::COLS;
            if (16 * j + i16 < pieces) {
#pragma unroll
                for (int e = 0; e < RP::COLS; e += 4)
                    *(float4*)(v + c0 + e) = float4{value(j, e), value(j, e + 1), value(j, e + 2), value(j, e + 3)};
            }
        }
    };
    auto chain = [&](const float* v) {
        RefAcc<OP> acc;
        int c = 0;
#pragma unroll 4
        for (; c + 4 <= d; c += 4) {
            const float4 x = *(const float4*)(v + c), y = *(const float4*)(qf + c);
            acc.add(y.x, x.x);
            acc.add(y.y, x.y);
            acc.add(y.z, x.z);
            acc.add(y.w, x.w);
        }
        for (; c < d; c++) acc.add(qf[c], v[c]);
        return acc.finish(sqn, sqd);
    };
    float s = 0.0f;
    if (OP == OP_DOT) {
        write_row(vals + g * P);
        __syncthreads();
        if (i16 == 0) s = chain(vals + g * P);
    } else {
        double sum = 0.0;
#pragma unroll
        for (int p = 0; p < RP::MAX; p++) {
            if (16 * p >= pieces) break;
            const int c0 = (16 * p + i16) * RP::COLS;
            if (16 * p + i16 < pieces) {
#pragma unroll
                for (int e = 0; e < RP::COLS; e++) {
                    const float q = qf[c0 + e], v = value(p, e);
                    const float x = OP == OP_COSINE ? v : fsub_rn(q, v);
                    const float y = OP == OP_COSINE ? q : x;
                    if (c0 + e < d) sum = __fma_rn((double)y, (double)x, sum);
                }
            }
        }
        sum = row16_dsum(sum);
        bool open = false;
        if (i16 == 0 && ok) {
            const double den = OP == OP_COSINE ? dmul_rn(sqn, sqd) : 0.0;
            // rounding errors of the two orders: at most d (sequential) and
            // d / 16 + 4 (lanes) steps of 2^-53 on the absolute terms' sum,
            // which is at most |q||d| (cosine) or the sum itself (l2); 5% over
            // for the bound's own roundings
            const double u = 1.1102230246251565e-16;
            const double terms = OP == OP_COSINE ? den : sum;
            const double err = 1.05 * u * (double)(d + d / 16 + 8) * terms + 1e-300;
            open = !ref_narrow<OP>(sum, err, den, s);
        }
        // undecided rows of this wave, one at a time through the wave's LDS row
        uint64_t left = __ballot(open);
        float* v = vals + (tid >> 6) * P;
        while (left) {
            const int l = __builtin_ctzll(left);
            left &= left - 1;
            if ((tid & 48) == (l & 48)) write_row(v);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if ((tid & 63) == l) s = chain(v);
            __builtin_amdgcn_wave_barrier();
        }
    }
    if (has && i16 == 0) keys[(int64_t)q0 * a.kp + at] = ok ? make_key(s, (uint32_t)cid, a.smallest) : 0ull;
}

// The same with a candidate a thread, grid (ceil(kp / 256), nq): one chain
// takes d dependent steps however few candidates there are, but every lane
// works, where above 15 of 16 wait for dot's chain or share a row's sum.
template <int FMT, int OP>
__global__ __launch_bounds__(256) void ref_rescore_rows_kernel(RefArgs a, uint64_t* __restrict__ keys) {
    __shared__ float qf[kMaxQueryDim];
    __shared__ double sqn_s;
    const int q = blockIdx.y, d = a.d;
    const int at = blockIdx.x * 256 + threadIdx.x;
    const bool has = at < a.kp;
    const int32_t cid = has ? a.cand_ids[(int64_t)q * a.kp + at] : -1;
    for (int c = threadIdx.x; c < d; c += 256) qf[c] = h2f(a.queries[(int64_t)q * d + c]);
    __syncthreads();
    // cosine: the query's norm, a sequential sum, on the last thread, while the
    // others sum their rows
    if (OP == OP_COSINE && threadIdx.x == 255) sqn_s = ref_sqrt_norm(qf, d);
    const bool ok = cid >= 0 && (int64_t)cid < a.n;
    const int64_t row = (int64_t)q * a.set_stride + (ok ? cid : 0);
    const double sqd = OP == OP_COSINE ? a.sqd[row] : 0.0;
    RefAcc<OP> acc;
    if (ok) {
        if (FMT == 8)
            acc = ref_acc_q8<OP>(qf, (const int8_t*)a.codes + row * a.pitch, ((const float*)a.scales)[row], d);
        else
            acc = ref_acc_q4<OP>(qf, (const uint8_t*)a.codes + row * a.pitch,
                                 (const uint16_t*)a.scales + row * (d / 32), d);
    }
    if (OP == OP_COSINE) __syncthreads();
    if (!has) return;
    const double sqn = OP == OP_COSINE ? sqn_s : 0.0;
    keys[(int64_t)q * a.kp + at] = ok ? make_key(acc.finish(sqn, sqd), (uint32_t)cid, a.smallest) : 0ull;
}

// ------------------------------------------------------- score matrix

// Reference scores of 256 / QG rows x QG * TQ queries a workgroup, each
// (row, query) pair the reference's own sequential chain: a thread owns one
// row and TQ queries.  KC columns of the rows at a time are dequantized into
// LDS (16-byte loads side by side, the next columns' in flight), the queries
// lie there whole; a piece of 4 columns feeds TQ chains from one LDS read of
// the row.  With a row per thread straight from memory the loads were 16 bytes
// out of every row, and every query read and dequantized the rows again: 8
// queries x 1,000 rows (d = 384, cosine) 36.5 us, now 12.5; 16 x 100,000
// 228, now 85.
template <int FMT, int OP, int QG, int TQ, int KC>
__global__ __launch_bounds__(256) void ref_scores_kernel(RefArgs a, int qtiles, float* __restrict__ out) {
    constexpr int RT = 256 / QG, NQ = QG * TQ;
    constexpr int LPR = FMT == 8 ? KC / 16 : KC / 32;          // 16-byte loads per row and stage
    constexpr int RPP = 256 / LPR;                             // rows per pass
    constexpr int NP = RT > RPP ? RT / RPP : 1;
    constexpr int COLS = KC / LPR;                             // columns per load
    constexpr int VP = KC + 4;
    extern __shared__ __attribute__((aligned(16))) float smem[];
    __shared__ double sqn_s[NQ];
    const int tid = threadIdx.x;
    const int d = a.d, dk = (d + KC - 1) / KC * KC;
    const int QP = dk + 4;
    float* vals = smem;             // [RT][VP]
    float* qf = smem + RT * VP;     // [NQ][QP]
    const int64_t rt = blockIdx.x / (unsigned)qtiles;
    const int q0 = (int)(blockIdx.x - rt * qtiles) * NQ + (int)blockIdx.y;  // (blockIdx.y: the set, one query each)
    const int nq = a.set_stride ? 1 : (a.nq - q0 < NQ ? a.nq - q0 : NQ);
    const int64_t r0 = rt * RT;
    const int64_t set_row0 = (int64_t)q0 * a.set_stride;
    const int lr = tid / LPR, lp = tid - lr * LPR;
    const int pieces = a.pitch / 16;

    v4i w[NP];
    float sc[NP];
    auto load = [&](int k0) {
        const int p = k0 / COLS + lp;
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int r = i * RPP + lr;
            const bool in = r < RT && r0 + r < a.n && p < pieces;
            const int64_t row = set_row0 + r0 + (in ? r : 0);
            w[i] = in ? *(const v4i*)((const uint8_t*)a.codes + row * a.pitch + 16 * p) : v4i{0, 0, 0, 0};
            sc[i] = !in ? 0.0f
                        : (FMT == 8 ? ((const float*)a.scales)[row] : h2f(((const uint16_t*)a.scales)[row * pieces + p]));
        }
    };
    load(0);
    for (int i = tid; i < NQ * dk; i += 256) {
        const int j = i / dk, c = i - j * dk;
        qf[j * QP + c] = j < nq && c < d ? h2f(a.queries[(int64_t)(q0 + j) * d + c]) : 0.0f;
    }
    if (OP == OP_COSINE) {
        // the queries' norms, 16 lanes each, while the first rows are in flight
        __syncthreads();
        for (int j = tid >> 4; j < NQ; j += 16) {
            const double v = ref_norm16(qf + j * QP, d);
            if ((tid & 15) == 0) sqn_s[j] = v;
        }
    }
    // thread: row tid / QG of the tile, queries qg, qg + QG, ...
    const int qg = tid % QG, r = tid / QG;
    const int64_t row = r0 + r;
    const double sqd = OP == OP_COSINE && row < a.n ? a.sqd[set_row0 + row] : 0.0;
    RefAcc<OP> acc[TQ];
    for (int k0 = 0; k0 < dk; k0 += KC) {
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int rr = i * RPP + lr;
            if (rr >= RT) continue;
            const int ws[4] = {w[i].x, w[i].y, w[i].z, w[i].w};
            float* dst = vals + rr * VP + lp * COLS;
            const int c0 = k0 + lp * COLS;
#pragma unroll
            for (int e = 0; e < COLS; e += 4) {
                float v[4];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const int x = e + u;
                    const int code = FMT == 8 ? (ws[x >> 2] << (24 - 8 * (x & 3))) >> 24 : (ws[x >> 3] << (28 - 4 * (x & 7))) >> 28;
                    v[u] = fmul_rn((float)code, sc[i]);
                    // columns past d: zeros whatever the scale (a sum is never
                    // -0, so adding 0 * 0 leaves it as it is)
                    if (FMT == 8 && c0 + x >= d) v[u] = 0.0f;
                }
                *(float4*)(dst + e) = float4{v[0], v[1], v[2], v[3]};
            }
        }
        __syncthreads();
        if (k0 + KC < dk) load(k0 + KC);
#pragma unroll 4
        for (int c = 0; c < KC; c += 4) {
            const float4 x4 = *(const float4*)(vals + r * VP + c);
            const float x[4] = {x4.x, x4.y, x4.z, x4.w};
#pragma unroll
            for (int j = 0; j < TQ; j++) {
                const float4 y4 = *(const float4*)(qf + (qg + j * QG) * QP + k0 + c);
                const float y[4] = {y4.x, y4.y, y4.z, y4.w};
#pragma unroll
                for (int u = 0; u < 4; u++) acc[j].add(y[u], x[u]);
            }
        }
        __syncthreads();
    }
    if (row >= a.n) return;
#pragma unroll
    for (int j = 0; j < TQ; j++) {
        const int lq = qg + j * QG;
        if (lq < nq) out[(int64_t)(q0 + lq) * a.n + row] = acc[j].finish(OP == OP_COSINE ? sqn_s[lq] : 0.0, sqd);
    }
}

// One workgroup per query: sort the candidates' reference keys, take the
// k-th, and prove (or not) from the scan score of the kp-th candidate that
// no other row reaches it.
template <int OP, int NT>
__global__ __launch_bounds__(NT) void ref_finish_kernel(RefArgs a, const uint64_t* __restrict__ cand_keys) {
    constexpr int NW = NT / 64;
    extern __shared__ uint64_t keys[];
    __shared__ float red_m[NW];
    __shared__ double red_g[NW], red_n[NW];
    __shared__ long long red_s[NW];
    __shared__ int ok_s;
    const int q = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int d = a.d;
    const uint16_t* qrow = a.queries + (int64_t)q * d;
    const int kp = a.kp;
    const int S = next_pow2(kp < 2 ? 2 : kp);
    for (int i = tid; i < S; i += NT) keys[i] = i < kp ? cand_keys[(int64_t)q * kp + i] : 0ull;

    // the quantities of the bounds: the scans' E16 codes of the query (same
    // arithmetic as encode_query_block), G = |q - qs*code|, |q|, sum code^2
    float m = 0.0f;
    for (int c = tid; c < d; c += NT) m = fmaxf(m, __builtin_fabsf(h2f(qrow[c])));
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    if (lane == 0) red_m[wave] = m;
    __syncthreads();
    float maxabs = 0.0f;
    for (int w = 0; w < NW; w++) maxabs = fmaxf(maxabs, red_m[w]);
    const float inv = maxabs == 0.0f ? 0.0f : fdiv_rn(32639.0f, maxabs);
    const float qs = maxabs == 0.0f ? 0.0f : fdiv_rn(maxabs, 32639.0f);
    double g2 = 0.0, n2 = 0.0;
    long long ss = 0;
    for (int c = tid; c < d; c += NT) {
        const float x = h2f(qrow[c]);
        const int code = maxabs != 0.0f ? code_e16(x, inv) : 0;
        const double diff = (double)x - (double)code * (double)qs;
        g2 += diff * diff;
        n2 += (double)x * (double)x;
        ss += (long long)code * code;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        g2 += __shfl_xor(g2, off);
        n2 += __shfl_xor(n2, off);
        ss += __shfl_xor(ss, off);
    }
    if (lane == 0) {
        red_g[wave] = g2;
        red_n[wave] = n2;
        red_s[wave] = ss;
    }
    __syncthreads();
    block_sort_desc_regs<NT>(keys, S);

    if (tid == 0) {
        const uint64_t kth = keys[a.k - 1];
        const float L = key_score(kth, a.smallest);
        bool ok = kth != 0;
        if (ok && (int64_t)kp < a.n) {
            if (maxabs == 0.0f && OP != OP_L2) {
                // a zero query: every reference dot / cosine is +0, as every
                // scan score, so the scan's first kp rows hold the k lowest
                ok = true;
            } else {
                const double up = 1.0 + 9.094947017729282e-13;
                double sg = 0.0, sn = 0.0;
                long long sc = 0;
                for (int w = 0; w < NW; w++) {
                    sg += red_g[w];
                    sn += red_n[w];
                    sc += red_s[w];
                }
                const double G = __builtin_sqrt(sg) * up;
                const double qn = __builtin_sqrt(sn) * up;
                const double qh = __builtin_sqrt((double)sc) * (double)qs * up;
                const double wide = 1.0 + 2.384185791015625e-07;  // 1 + 2^-22
                const RefBounds b = ref_bounds(OP, G, qn, qh, (double)a.e_qd, (double)a.maxdn * wide,
                                               (double)a.maxdd * wide, d);
                const double c = (double)a.cand_scores[(int64_t)q * kp + kp - 1];
                ok = b.ok && (a.smallest ? ref_lo(b, c) > (double)L : ref_hi(b, c) < (double)L);
            }
        }
        ok_s = ok ? 1 : 0;
        a.redo[q] = ok ? 0 : 1;
        // every key of the final k is at least kth, hence at least the
        // smallest key of its score (low word 0x7FFFFFFF is below every ~idx)
        a.redo_tau[q] = kth ? make_key(L, 0x80000000u, a.smallest) : 0ull;
    }
    __syncthreads();
    if (!ok_s) return;
    for (int i = tid; i < a.k; i += NT) {
        const uint64_t key = keys[i];
        a.out_ids[(int64_t)q * a.k + i] = key ? (int32_t)key_index(key) : -1;
        if (a.out_scores) a.out_scores[(int64_t)q * a.k + i] = key ? key_score(key, a.smallest) : 0.0f;
    }
}

// Reference scores of every row, lane = row.  Score matrix (a.out_scores):
// grid (parts, nq), one query per blockIdx.y.  Top-k: grid (parts, R); the
// workgroups of blockIdx.y = r take the queries r, r + R, ... the finish
// marked (redo == nullptr: all of them), each with the streaming reservoir
// from the threshold key redo_tau and the last-workgroup merge over the
// gridDim.x parts.  A query nobody marked costs its workgroups one flag read.
template <int FMT, int OP>
__global__ __launch_bounds__(256) void ref_scan_kernel(ScanArgs a, int nq, const double* __restrict__ sqd,
                                                       const int* __restrict__ redo,
                                                       const uint64_t* __restrict__ redo_tau) {
    extern __shared__ uint64_t topk_keys[];
    __shared__ ScanTopkLds S;
    __shared__ float qf[kMaxQueryDim];
    __shared__ double sqn_s;
    __shared__ int marked[256];
    __shared__ int nmarked;
    const bool topk = a.out_scores == nullptr;
    // this slot's queries, 256 at a time: the marks are read in parallel and
    // the marked queries listed in LDS (the list is usually empty)
    const int per_slot = (nq - (int)blockIdx.y + (int)gridDim.y - 1) / (int)gridDim.y;
    for (int base = 0; base < per_slot; base += 256) {
        __syncthreads();  // the previous batch's list is consumed
        if (threadIdx.x == 0) nmarked = 0;
        __syncthreads();
        {
            const int j = base + (int)threadIdx.x;
            const int qj = (int)blockIdx.y + j * (int)gridDim.y;
            if (j < per_slot && (!topk || !redo || redo[qj])) marked[atomicAdd(&nmarked, 1)] = qj;
        }
        __syncthreads();
        const int nm = nmarked;
        for (int mi = 0; mi < nm; mi++) {
            const int qi = marked[mi];
            const uint64_t tau0 = (topk && redo_tau) ? redo_tau[qi] : 0ull;
            __syncthreads();  // the previous query's readers of qf and the reservoir are done
            const uint16_t* qrow = a.queries + (int64_t)qi * a.d;
            for (int c = threadIdx.x; c < a.d; c += 256) qf[c] = h2f(qrow[c]);
            __syncthreads();
            if (OP == OP_COSINE && threadIdx.x == 0) sqn_s = ref_sqrt_norm(qf, a.d);
            if (topk) topk_init(topk_keys, &S.st);  // (its barrier publishes sqn_s)
            else __syncthreads();
            const double sqn = OP == OP_COSINE ? sqn_s : 0.0;
            const int64_t set_row0 = (int64_t)qi * a.set_stride;
            const int64_t wg_row0 = (int64_t)blockIdx.x * a.rounds * 256;
            for (int r = 0; r < a.rounds; r++) {
                const int64_t row = wg_row0 + (int64_t)r * 256 + threadIdx.x;
                const bool valid = row < a.n;
                float s = 0.0f;
                if (valid)
                    s = ref_row_score<FMT, OP>(a.codes, a.scales, sqd, set_row0 + row, a.pitch, a.d, qf, sqn);
                if (!topk) {
                    if (valid) a.out_scores[(int64_t)qi * a.n + row] = s;
                    continue;
                }
                const uint64_t key = valid ? make_key(s, (uint32_t)row, a.smallest) : 0ull;
                const uint64_t tau = S.st.tau > tau0 ? S.st.tau : tau0;
                topk_offer(key, tau, topk_keys, &S.st);
                if (a.mid_compact) {
                    __syncthreads();
                    topk_maybe_compact(topk_keys, &S.st, a.k, a.cap);
                }
            }
            if (topk) finish_topk(a, topk_keys, S, qi);
        }
    }
}

// ----------------------------------------------------------------- hosts

static int next_pow2_host(int x) {
    int p = 2;
    while (p < x) p <<= 1;
    return p;
}

// Candidates past which a row a thread is faster (us, 16 lanes a row / a row a
// thread, by candidates in all):
//              q8 d 64   384      1,000       q4 d 128  384      1,024
//   dot    3K  7 / 7    12 / 19  24 / 42      7 / 6   12 / 10   24 / 18
//         26K  7 / 7    19 / 20  56 / 45     10 / 6   21 / 10   60 / 21
//        309K 31 / 16  125 / 45 429 / 115    52 / 13 141 / 39  480 / 102
//   cosine 7K  7 / 7     8 / 21  10 / 48      7 / 7    8 / 11   11 / 23
//         26K 10 / 9    12 / 24  23 / 54     10 / 8   13 / 15   25 / 31
//         80K 19 / 9    25 / 23  39 / 48     20 / 9   27 / 16   46 / 32
//   l2    26K  8 / 8    10 / 22  16 / 48      8 / 7   10 / 12   16 / 23
//         80K 13 / 9    19 / 24  30 / 49     15 / 9   22 / 16   35 / 30
//        309K 37 / 17   55 / 49 104 / 114    43 / 17  67 / 43  117 / 111
// (q8's row a thread reads 16 bytes out of every row per load, so wide rows
// hold it back; q4 rows are half as long)
template <int FMT, int OP>
static int64_t ref_rescore_few(int d) {
    if (OP == OP_DOT) return FMT == 8 ? 24 * 1024 : 0;
    if (FMT == 8) return (OP == OP_COSINE ? 200 : 400) * (int64_t)d;
    return OP == OP_COSINE ? 28 * 1024 : 40 * 1024;
}

template <int FMT, int OP>
static hipError_t launch_ref_rescore_op(const RefArgs& a, uint64_t* keys, hipStream_t s) {
    if ((int64_t)a.nq * a.kp > ref_rescore_few<FMT, OP>(a.d)) {
        const dim3 grid((unsigned)((a.kp + 255) / 256), (unsigned)a.nq);
        hipLaunchKernelGGL((ref_rescore_rows_kernel<FMT, OP>), grid, dim3(256), 0, s, a, keys);
        return hipGetLastError();
    }
    const dim3 grid((unsigned)((a.kp + 15) / 16), (unsigned)a.nq);
    const size_t lds = (size_t)(1 + (OP == OP_DOT ? 16 : 4)) * ref_row_pitch(a.d) * sizeof(float);
    hipLaunchKernelGGL((ref_rescore_kernel<FMT, OP>), grid, dim3(256), lds, s, a, keys);
    return hipGetLastError();
}

template <int FMT>
static hipError_t launch_ref_rescore_fmt(const RefArgs& a, uint64_t* keys, hipStream_t s) {
    switch (a.op) {
        case OP_DOT: return launch_ref_rescore_op<FMT, OP_DOT>(a, keys, s);
        case OP_COSINE: return launch_ref_rescore_op<FMT, OP_COSINE>(a, keys, s);
        default: return launch_ref_rescore_op<FMT, OP_L2>(a, keys, s);
    }
}

hipError_t launch_ref_rescore(const RefArgs& a, uint64_t* keys, hipStream_t s) {
    if (a.d <= 0 || a.d > kMaxQueryDim || a.kp <= 0 || a.nq <= 0 || a.nq > 65535) return hipErrorInvalidValue;
    if (a.fmt == 4 && a.d % 32 != 0) return hipErrorInvalidValue;
    return a.fmt == 8 ? launch_ref_rescore_fmt<8>(a, keys, s) : launch_ref_rescore_fmt<4>(a, keys, s);
}

template <int FMT, int OP, int QG, int TQ, int KC>
static hipError_t launch_ref_scores_tile(const RefArgs& a, float* out, hipStream_t s) {
    constexpr int RT = 256 / QG, NQ = QG * TQ;
    const int64_t rtiles = (a.n + RT - 1) / RT;
    const int qtiles = a.set_stride ? 1 : (a.nq + NQ - 1) / NQ;
    if (rtiles * qtiles > 0x7FFFFFFF) return hipErrorInvalidValue;
    const int dk = (a.d + KC - 1) / KC * KC;
    const size_t lds = ((size_t)RT * (KC + 4) + (size_t)NQ * (dk + 4)) * sizeof(float);
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute((const void*)ref_scores_kernel<FMT, OP, QG, TQ, KC>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    const dim3 grid((unsigned)(rtiles * qtiles), a.set_stride ? (unsigned)a.nq : 1u);
    hipLaunchKernelGGL((ref_scores_kernel<FMT, OP, QG, TQ, KC>), grid, dim3(256), lds, s, a, qtiles, out);
    return hipGetLastError();
}

// The tile, from the queries that share the rows.  More chains a thread read
// and convert a row's columns once for several queries, but need enough pairs
// to fill the chip (us, d = 384 unless said; the rows per workgroup are 256
// over the first number):
//                               8x1 KC128   4x4 KC64   4x2 KC64   4x1 KC64   1x1 KC32
//   16 x 100,000 cosine q8            108         85
//   100 x 1,000 cosine q8            15.2       23.1
//   8 x 100,000 cosine q8            60.5                  53.1
//   8 x 1,000 cosine q8              12.5                  16.3
//   4 x 5,000 cosine q8                                    16.5       12.4       24
//   1 x 1,000 l2 q8, d = 128                                           5.8      7.6
//   1 x 1,000,000 cosine q8, d = 128                                    98       52
template <int FMT, int OP>
static hipError_t launch_ref_scores_op(const RefArgs& a, float* out, hipStream_t s) {
    const int nq = a.set_stride ? 1 : a.nq;
    const bool few = a.n * nq < 512 * 1024;
    // (16 queries of rows past 960 columns hold over half a CU's 160 KB of LDS:
    // two tiles of 8 instead.  10 q4 queries x 118,304 x 1,024, dot: 334 us, now
    // 175; 11 q8 queries x 546,039 x 768, cosine: 827, and 887 as two tiles)
    if (nq > 8 && !few && a.d <= 960) return launch_ref_scores_tile<FMT, OP, 4, 4, 64>(a, out, s);
    if (nq > 4 && !few) return launch_ref_scores_tile<FMT, OP, 4, 2, 64>(a, out, s);
    // (stages of 128 columns would be half empty at the end of these rows)
    if (nq > 4 && ((a.d + 63) / 64) % 2 != 0) return launch_ref_scores_tile<FMT, OP, 8, 1, 64>(a, out, s);
    if (nq > 4) return launch_ref_scores_tile<FMT, OP, 8, 1, 128>(a, out, s);
    const int64_t rows = a.set_stride ? a.n * a.nq : a.n;
    if (nq > 1 || rows < 64 * 1024) return launch_ref_scores_tile<FMT, OP, 4, 1, 64>(a, out, s);
    return launch_ref_scores_tile<FMT, OP, 1, 1, 32>(a, out, s);
}

template <int FMT>
static hipError_t launch_ref_scores_fmt(const RefArgs& a, float* out, hipStream_t s) {
    switch (a.op) {
        case OP_DOT: return launch_ref_scores_op<FMT, OP_DOT>(a, out, s);
        case OP_COSINE: return launch_ref_scores_op<FMT, OP_COSINE>(a, out, s);
        default: return launch_ref_scores_op<FMT, OP_L2>(a, out, s);
    }
}

hipError_t launch_ref_scores(const RefArgs& a, float* out, hipStream_t s) {
    if (a.d <= 0 || a.d > kMaxQueryDim || a.nq <= 0 || a.pitch % 16 != 0) return hipErrorInvalidValue;
    if (a.fmt == 4 && (a.d % 32 != 0 || a.pitch != a.d / 2)) return hipErrorInvalidValue;
    return a.fmt == 8 ? launch_ref_scores_fmt<8>(a, out, s) : launch_ref_scores_fmt<4>(a, out, s);
}

hipError_t launch_ref_finish(const RefArgs& a, const uint64_t* keys, hipStream_t s) {
    if (a.d <= 0 || a.d > kMaxQueryDim || a.k <= 0 || a.kp < a.k || a.nq <= 0) return hipErrorInvalidValue;
    const int S = next_pow2_host(a.kp);
    if (S > kRefMaxKeys) return hipErrorInvalidValue;
    const size_t lds = (size_t)S * 8;
    const dim3 grid((unsigned)a.nq);
    // 1024 threads sort the larger candidate sets (fewer register slots and
    // network steps per thread)
    if (S > 512) {
        switch (a.op) {
            case OP_DOT: hipLaunchKernelGGL((ref_finish_kernel<OP_DOT, 1024>), grid, dim3(1024), lds, s, a, keys); break;
            case OP_COSINE:
                hipLaunchKernelGGL((ref_finish_kernel<OP_COSINE, 1024>), grid, dim3(1024), lds, s, a, keys);
                break;
            default: hipLaunchKernelGGL((ref_finish_kernel<OP_L2, 1024>), grid, dim3(1024), lds, s, a, keys); break;
        }
    } else {
        switch (a.op) {
            case OP_DOT: hipLaunchKernelGGL((ref_finish_kernel<OP_DOT, 256>), grid, dim3(256), lds, s, a, keys); break;
            case OP_COSINE:
                hipLaunchKernelGGL((ref_finish_kernel<OP_COSINE, 256>), grid, dim3(256), lds, s, a, keys);
                break;
            default: hipLaunchKernelGGL((ref_finish_kernel<OP_L2, 256>), grid, dim3(256), lds, s, a, keys); break;
        }
    }
    return hipGetLastError();
}

template <int FMT>
static hipError_t launch_ref_scan_fmt(int op, const ScanArgs& a, int nq, const double* sqd, const int* redo,
                                      const uint64_t* redo_tau, dim3 grid, size_t lds, hipStream_t s) {
    const dim3 block(256);
    switch (op) {
        case OP_DOT:
            hipLaunchKernelGGL((ref_scan_kernel<FMT, OP_DOT>), grid, block, lds, s, a, nq, sqd, redo, redo_tau);
            break;
        case OP_COSINE:
            hipLaunchKernelGGL((ref_scan_kernel<FMT, OP_COSINE>), grid, block, lds, s, a, nq, sqd, redo, redo_tau);
            break;
        default:
            hipLaunchKernelGGL((ref_scan_kernel<FMT, OP_L2>), grid, block, lds, s, a, nq, sqd, redo, redo_tau);
            break;
    }
    return hipGetLastError();
}

hipError_t launch_ref_scan(int fmt, int op, const ScanArgs& a, int nq, const double* sqd, const int* redo,
                           const uint64_t* redo_tau, dim3 grid, size_t lds, hipStream_t s) {
    if (a.d <= 0 || a.d > kMaxQueryDim || nq <= 0) return hipErrorInvalidValue;
    if (fmt == 4 && a.d % 32 != 0) return hipErrorInvalidValue;
    return fmt == 8 ? launch_ref_scan_fmt<8>(op, a, nq, sqd, redo, redo_tau, grid, lds, s)
                    : launch_ref_scan_fmt<4>(op, a, nq, sqd, redo, redo_tau, grid, lds, s);
}

}  // namespace manta
