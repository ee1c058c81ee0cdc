// kernels_score.hip -- packed-candidate scoring for gfx950 (streaming path).
//
// One launch per fused score+top-k call.  Each workgroup (256 threads, 4
// waves) scores `rounds` x 256 candidate rows against one query.  q8 rows
// are read with coalesced 16-byte buffer loads: L lanes cover one row (L*16
// contiguous bytes per load), C loads per lane per row, so a wave moves
// 64*16 bytes per load instruction.  The int8 products run on v_dot4 with
// the query codes held in registers (each lane encodes the columns it
// multiplies); a DPP group sum over the L lanes leaves every lane of a group
// the row total, and lane g*L + j keeps row g*L + j, so after a round each
// lane owns one row for the epilogue.  The epilogue computes the f32 score
// and either stores it (score matrix), offers its key to per-wave sorted
// register lists (small k, and up to 64 with too many parts for the next),
// keeps it in LDS for a selection at the end (k <= kBestMaxK), or offers its
// key to the LDS reservoir.  In top-k mode each workgroup publishes its k best keys; the last workgroup of a query (atomic
// ticket) merges them into the final ids.
//
// Quantized-query scores (the CPU oracle restates them):
//   q8 dot    (E8 query codes):  t = s_r*acc; t = t*qmax; score = t/127
//             (BASELINE's q8 dot formula, the quantized-query dot);
//   q8 E16 codes (hi/lo digits): qd = (s_r*qs)*f32(acc); dot16 = qd;
//             cosine = den == 0 ? 0 : qd/den with den = |q|*|d_r|;
//             l2 = sqrt(max(0, (qq + dd_r) - 2*qd));
//   q4        (E16):             qd = qs * fma-chain over blocks of
//                                f16scale_b * f32(acc_b); then as above.
// The E16 scores rank rows for the reference-semantics top-k, which
// rescores the best of them with the reference's arithmetic
// (kernels_ref.hip).
#include "best_common.hpp"
#include "device_common.hpp"
#include "kernels.hpp"
#include "q4_common.hpp"
#include "scan_common.hpp"

namespace manta {

// ------------------------------------------------------------ query codes

// q4 digit planes are permuted per 8 columns to [c0 c2 c4 c6 c1 c3 c5 c7]
// so that the nibble unpack below feeds v_dot4 without shuffling.
__device__ __forceinline__ int q4_perm_pos(int c) {
    const int j = c & 7;
    return (c & ~7) + ((j & 1) ? 4 + (j >> 1) : (j >> 1));
}

enum { ENC_E8 = 0, ENC_E16 = 1, ENC_E16_Q4 = 2 };

struct QueryLds {
    int8_t c8[kMaxQueryDim];
    int8_t hi[kMaxQueryDim];
    int8_t lo[kMaxQueryDim];
    QConst qc;
    float redf[4];
    long long redi[4];
};

// Encode one f16 query into LDS (whole workgroup, 256 threads).  `span` is
// the number of code slots to fill (the row pitch; columns >= d get 0).
__device__ inline void encode_query_block(const uint16_t* __restrict__ qrow, int d, int span, int enc,
                                          QueryLds& L) {
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    float m = 0.0f;
    for (int c = tid; c < d; c += 256) m = fmaxf(m, __builtin_fabsf(h2f(qrow[c])));
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    if (lane == 0) L.redf[wave] = m;
    __syncthreads();
    const float maxabs = fmaxf(fmaxf(L.redf[0], L.redf[1]), fmaxf(L.redf[2], L.redf[3]));
    if (enc == ENC_E8) {
        const float qmax = fmaxf(1.0f, maxabs);
        for (int c = tid; c < span; c += 256) L.c8[c] = (int8_t)(c < d ? code_e8(h2f(qrow[c]), qmax) : 0);
        if (tid == 0) L.qc = QConst{qmax, 0.0f, 0.0f, 0.0f};
        __syncthreads();
        return;
    }
    const float inv = maxabs == 0.0f ? 0.0f : fdiv_rn(32639.0f, maxabs);
    long long ss = 0;
    for (int c = tid; c < span; c += 256) {
        const int code = (c < d && maxabs != 0.0f) ? code_e16(h2f(qrow[c]), inv) : 0;
        const int l = (int)(int8_t)(code & 0xFF);
        const int h = (code - l) >> 8;
        const int pos = enc == ENC_E16_Q4 ? q4_perm_pos(c) : c;
        L.hi[pos] = (int8_t)h;
        L.lo[pos] = (int8_t)l;
        ss += (long long)code * code;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) ss += __shfl_xor(ss, off);
    if (lane == 0) L.redi[wave] = ss;
    __syncthreads();
    if (tid == 0) L.qc = e16_consts(maxabs, L.redi[0] + L.redi[1] + L.redi[2] + L.redi[3]);
    __syncthreads();
}

// Global-memory variant: one workgroup per query (used by the batched
// paths, whose many workgroups share each query).
__global__ __launch_bounds__(256) void query_encode_kernel(const uint16_t* __restrict__ q, int d, int pitch,
                                                           int e16, int8_t* __restrict__ c8,
                                                           int8_t* __restrict__ hi, int8_t* __restrict__ lo,
                                                           QConst* __restrict__ qc, uint64_t* __restrict__ tau,
                                                           int* __restrict__ bcnt) {
    __shared__ QueryLds L;
    const int qi = blockIdx.x;
    // e16: 0 = E8 codes, 1 = E16 digit planes, 2 = E16 planes in the q4 nibble order
    encode_query_block(q + (int64_t)qi * d, d, pitch, e16 == 2 ? ENC_E16_Q4 : (e16 ? ENC_E16 : ENC_E8), L);
    for (int c = threadIdx.x; c < pitch; c += 256) {
        if (e16) {
            hi[(int64_t)qi * pitch + c] = L.hi[c];
            lo[(int64_t)qi * pitch + c] = L.lo[c];
        } else {
            c8[(int64_t)qi * pitch + c] = L.c8[c];
        }
    }
    if (threadIdx.x == 0) {
        qc[qi] = L.qc;
        // the threshold passes start from no threshold and no kept keys
        if (tau) tau[qi] = 0ull;
        if (bcnt) bcnt[qi] = 0;
    }
}

// Shadow-scan query encoding (one workgroup per query): the E16 planes in
// the q4 order and constants as above, full-range int8 codes
// c = round(q * 127/maxabs) with qa = maxabs/127 for the shadow's A operand,
// and shadow_bound's margin m and factor f.  With q^ the E16-dequantized
// query and G = |q^ - qa c|, a row's exact score and its shadow pre-score
// p differ by at most E/|x| + (F/|x|) G/|q^| (cosine, in score units; p
// scaled by f = |q^|/qa) or E|q^| + F G (dot, f = 1/qa), E and F the
// shadow's row error terms (ShadowInfo maxima); m adds 2^-16 (times the
// largest |x||q^| for dot), far above every f32 rounding on either side.
__global__ __launch_bounds__(256) void query_encode_shadow_kernel(const uint16_t* __restrict__ q, int d, int spitch,
                                                                  int op, const ShadowInfo* __restrict__ info,
                                                                  int8_t* __restrict__ c8, int8_t* __restrict__ hi,
                                                                  int8_t* __restrict__ lo, QConst* __restrict__ qc,
                                                                  float* __restrict__ qb, uint64_t* __restrict__ tau,
                                                                  int* __restrict__ bcnt) {
    __shared__ QueryLds L;
    __shared__ double g2s[4];
    __shared__ long long sss[4];
    const int qi = blockIdx.x;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const uint16_t* qrow = q + (int64_t)qi * d;
    encode_query_block(qrow, d, d, ENC_E16_Q4, L);
    const float maxabs = fmaxf(fmaxf(L.redf[0], L.redf[1]), fmaxf(L.redf[2], L.redf[3]));
    const float qs = L.qc.a;
    const float inv16 = maxabs == 0.0f ? 0.0f : fdiv_rn(32639.0f, maxabs);
    const float qa = fdiv_rn(maxabs, 127.0f);
    const float inv8 = maxabs == 0.0f ? 0.0f : fdiv_rn(127.0f, maxabs);
    double g2 = 0.0;
    long long ss = 0;
    for (int c = tid; c < spitch; c += 256) {
        int k8 = 0;
        if (c < d && maxabs != 0.0f) {
            const float x = h2f(qrow[c]);
            k8 = (int)fminf(127.0f, fmaxf(-127.0f, round_half_away(fmul_rn(x, inv8))));
            const int k16 = code_e16(x, inv16);
            const double diff = (double)k16 * (double)qs - (double)k8 * (double)qa;
            g2 += diff * diff;
            ss += (long long)k16 * k16;
        }
        c8[(int64_t)qi * spitch + c] = (int8_t)k8;
    }
    for (int c = tid; c < d; c += 256) {
        hi[(int64_t)qi * d + c] = L.hi[c];
        lo[(int64_t)qi * d + c] = L.lo[c];
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        g2 += __shfl_xor(g2, off);
        ss += __shfl_xor(ss, off);
    }
    if (lane == 0) {
        g2s[wave] = g2;
        sss[wave] = ss;
    }
    __syncthreads();
    if (tid == 0) {
        qc[qi] = L.qc;
        if (tau) tau[qi] = 0ull;
        if (bcnt) bcnt[qi] = 0;
        const double G = __builtin_sqrt(g2s[0] + g2s[1] + g2s[2] + g2s[3]);
        const double qn = __builtin_sqrt((double)(sss[0] + sss[1] + sss[2] + sss[3])) * (double)qs;
        const double up = 1.0 + 9.5367431640625e-7;
        float m = 0.0f, f = 0.0f;
        if (qn > 0.0) {
            const double me_c = __uint_as_float(info->me_cos), mf_c = __uint_as_float(info->mf_cos);
            const double me_d = __uint_as_float(info->me_dot), mf_d = __uint_as_float(info->mf_dot);
            const double mn = __uint_as_float(info->maxn);
            if (op == OP_COSINE) {
                m = (float)((me_c + mf_c * G / qn + 1.52587890625e-05) * up);
                f = (float)(qn / (double)qa);
            } else {
                m = (float)((me_d * qn + mf_d * G + 1.52587890625e-05 * mn * qn) * up);
                f = (float)(1.0 / (double)qa);
            }
        }
        qb[2 * qi] = m;
        qb[2 * qi + 1] = f;
    }
}

// ----------------------------------------------------------- epilogues

template <int OP>
__device__ __forceinline__ float q8_epilogue(int acc_or_hi, int lo, float scale, const QConst& k,
                                             float dnorm, float dd) {
    if (OP == OP_DOT) {
        float t = fmul_rn(scale, (float)acc_or_hi);
        t = fmul_rn(t, k.a);
        return fdiv_rn(t, 127.0f);
    }
    // f32(256*hi + lo) with one rounding: both terms are exact in f32.
    float dotf = __fmaf_rn(256.0f, (float)acc_or_hi, (float)lo);
    float qd = fmul_rn(fmul_rn(scale, k.a), dotf);
    if (OP == OP_DOT16) return qd;
    if (OP == OP_COSINE) {
        float den = fmul_rn(k.b, dnorm);
        return den == 0.0f ? 0.0f : fdiv_rn(qd, den);
    }
    float t = fadd_rn(k.c, dd);
    float dist2 = fsub_rn(t, fmul_rn(2.0f, qd));
    dist2 = dist2 < 0.0f ? 0.0f : dist2;
    return fsqrt_rn(dist2);
}

__device__ __forceinline__ int dot16(v4i a, v4i b, int acc) {
    acc = __builtin_amdgcn_sdot4(a.x, b.x, acc, false);
    acc = __builtin_amdgcn_sdot4(a.y, b.y, acc, false);
    acc = __builtin_amdgcn_sdot4(a.z, b.z, acc, false);
    acc = __builtin_amdgcn_sdot4(a.w, b.w, acc, false);
    return acc;
}

// ------------------------------------------------------- top-k plumbing

struct ScanLds {
    QueryLds q;
    TopKShared st;
    int last;
};

// One round's score of this thread's row (round r of the workgroup): stored,
// buffered for finish_buffered, or offered to the reservoir.
__device__ __forceinline__ void emit_round(const ScanArgs& a, float score, bool valid, int64_t row, int r, int qi,
                                           uint64_t* keys, TopKShared* st) {
    if (a.out_scores) {
        if (valid) a.out_scores[(int64_t)qi * a.n + row] = score;
        return;
    }
    if (a.buffered) {
        const uint32_t o = float_order(score);
        ((uint32_t*)keys)[r * 256 + threadIdx.x] = valid ? (a.smallest ? ~o : o) : 0u;
        return;
    }
    const uint64_t key = valid ? make_key(score, (uint32_t)row, a.smallest) : 0ull;
    topk_offer(key, st->tau, keys, st);
    if (a.mid_compact) {
        __syncthreads();
        topk_maybe_compact(keys, st, a.k, a.cap);
    }
}

// End of a buffered top-k scan workgroup (k <= kBestMaxK; on the fixed-width
// q8 kernel, k past the wave lists'): its scores are in LDS, a thread's own
// rows in its own words, so the rounds ran without a barrier or an atomic; the
// k best of them, and of the query's parts, by a floor and ranks.  Against the
// reservoir (compactions between rounds, the
// last workgroup streaming every part key through it): one q4 query, 1,048,576
// rows, k = 108, 159 -> 65 us.
__device__ __forceinline__ void finish_buffered(const ScanArgs& a, const uint64_t* buf, int qi) {
    __shared__ BestShared B;
    const uint32_t* slots = (const uint32_t*)buf;  // (rows past n: 0)
    const int tid = threadIdx.x;
    const int64_t row0 = (int64_t)blockIdx.x * a.rounds * 256;
    const int left = a.n - row0 < (int64_t)a.rounds * 256 ? (int)(a.n - row0) : a.rounds * 256;
    int kept = block_best<0>([&](int j) { return slots[j * 256 + tid]; },
                             [&](int j) { return j * 256 + tid < left ? (int)(row0 + j * 256 + tid) : -1; }, a.rounds,
                             a.k, B);
    if (kept < 0)
        kept = best_streamed([&](int64_t i) { return ((uint64_t)slots[i] << 32) | (uint64_t)(~(uint32_t)(row0 + i)); },
                             left, 1ull, a.k, B);
    if (gridDim.x > 1) {
        kept = merge_best_parts(a.partial, a.tickets, qi, kept, a.k, B);
        if (kept < 0) return;
    }
    for (int i = tid; i < a.k; i += 256) {
        const uint64_t e = i < kept ? B.keys[i] : 0ull;
        a.out_ids[(int64_t)qi * a.k + i] = e ? (int32_t)key_index(e) : -1;
        if (a.out_topk_scores) a.out_topk_scores[(int64_t)qi * a.k + i] = e ? key_score(e, a.smallest) : 0.0f;
    }
}

// End of a top-k scan workgroup on the wave-list path (k <= 64): the waves'
// lists merge into wave 0's, which publishes the workgroup's k best keys
// (sorted) as finish_topk does; the last workgroup of the query merges all
// parts with the same lists, 8 keys per lane in flight, and writes ids and
// scores straight from wave 0's lanes.  buf: blockDim.x keys of LDS.
template <class SL>
__device__ inline void finish_wave_lists(const ScanArgs& a, uint64_t list, uint64_t thr, uint64_t* buf, SL& S,
                                         int qi) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    wave_lists_merge(list, thr, a.k, buf);
    const int64_t per_q = (int64_t)gridDim.x * a.k;
    uint64_t* dst = a.partial + (int64_t)qi * per_q + (int64_t)blockIdx.x * a.k;
    if (wave == 0 && lane < a.k) __hip_atomic_store(dst + lane, list, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // Publication order at the ISA level (gfx950): every access to the parts
    // and the ticket is an agent-scope atomic, which the AMDGPU memory model
    // implements as sc1 accesses performed at the device coherence point
    // (past the per-XCD L2s); s_waitcnt vmcnt(0) retires this wave's part
    // stores there before the barrier, the ticket RMW is issued after it,
    // and the last workgroup's sc1 loads read the coherence point.  A
    // source-level release/acquire pair would add an L2 writeback per
    // workgroup (buffer_wbl2): 11% more time on a 32-problem q8 scan.
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0)
        S.last = __hip_atomic_fetch_add(&a.tickets[qi], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                 gridDim.x - 1;
    __syncthreads();
    if (!S.last) return;
    const uint64_t* src = a.partial + (int64_t)qi * per_q;
    // Up to one part key per thread (C0's 32-problem launch: 8 parts of 10):
    // every key counts the keys above it and the k best land at their ranks,
    // no insertions on the launch's last step.
    if (per_q <= (int64_t)blockDim.x) {
        __shared__ uint64_t res[64];  // k <= 64 on the list path
        const int t = (int)threadIdx.x, n = (int)per_q, k = a.k;
        const uint64_t mine = t < n ? __hip_atomic_load(src + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
        buf[t] = mine;
        if (t < 64) res[t] = 0ull;
        __syncthreads();
        int rank = 0;
        if (mine)
            for (int i = 0; i < n; i++) rank += buf[i] > mine ? 1 : 0;
        if (mine && rank < k) res[rank] = mine;  // keys are distinct: so are their ranks
        __syncthreads();
        if (t < k) {
            const uint64_t key = res[t];
            a.out_ids[(int64_t)qi * k + t] = key ? (int32_t)key_index(key) : -1;
            if (a.out_topk_scores) a.out_topk_scores[(int64_t)qi * k + t] = key ? key_score(key, a.smallest) : 0.0f;
        }
        if (t == 0) __hip_atomic_store(&a.tickets[qi], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    // Many parts (a single query's call: 128 parts of k): the k-th largest
    // part head is a floor of the final k-th key (the k best heads are k
    // distinct keys), only the k parts whose heads reach it hold keys at or
    // above it, and those k^2 or fewer candidates take their place by rank
    // (each counts the candidates above it) instead of one insertion each.
    // Fewer than k keys in the parts' heads: the lists below.
    if (a.k <= 16 && (int)gridDim.x >= a.k && gridDim.x <= 256) {
        __shared__ uint64_t heads[256];
        __shared__ uint64_t floor_s;
        __shared__ int ncand;
        const int t = (int)threadIdx.x, P = (int)gridDim.x, k = a.k;
        uint64_t mk[16];
#pragma unroll
        for (int j = 0; j < 16; j++)
            mk[j] = (t < P && j < k) ? __hip_atomic_load(src + (int64_t)t * k + j, __ATOMIC_RELAXED,
                                                          __HIP_MEMORY_SCOPE_AGENT)
                                     : 0ull;
        heads[t] = mk[0];  // a part's list is sorted: its first key is its best
        if (t == 0) {
            floor_s = 0ull;
            ncand = 0;
        }
        __syncthreads();
        if (t < P && mk[0]) {
            int rank = 0;
            for (int i = 0; i < P; i++) rank += heads[i] > mk[0] ? 1 : 0;
            if (rank == k - 1) floor_s = mk[0];  // keys are distinct: one thread
        }
        __syncthreads();
        const uint64_t fl = floor_s;
        if (fl) {
            int cnt = 0;
#pragma unroll
            for (int j = 0; j < 16; j++) cnt += mk[j] >= fl ? 1 : 0;  // (empty slots are 0 < fl)
            if (t < P && cnt) {
                int pos = atomicAdd(&ncand, cnt);
#pragma unroll
                for (int j = 0; j < 16; j++)
                    if (mk[j] >= fl) buf[pos++] = mk[j];
            }
            __syncthreads();
            const int nc = ncand;  // k <= nc <= k^2 <= blockDim.x
            const uint64_t mine = t < nc ? buf[t] : 0ull;
            int rank = 0;
            if (t < nc)
                for (int i = 0; i < nc; i++) rank += buf[i] > mine ? 1 : 0;
            __syncthreads();  // every read of buf is done
            if (t < nc && rank < k) buf[rank] = mine;
            __syncthreads();
            if (t < k) {
                const uint64_t key = buf[t];
                a.out_ids[(int64_t)qi * k + t] = (int32_t)key_index(key);
                if (a.out_topk_scores) a.out_topk_scores[(int64_t)qi * k + t] = key_score(key, a.smallest);
            }
            if (t == 0) __hip_atomic_store(&a.tickets[qi], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return;
        }
    }
    list = 0;
    thr = 0;
    // batches of 64 keys go to the waves in turn; B batches per wave in flight
    constexpr int B = 8;
    const int64_t stride = (int64_t)blockDim.x;
    for (int64_t base = (int64_t)wave * 64; base < per_q; base += stride * B) {
        uint64_t kb[B];
#pragma unroll
        for (int b = 0; b < B; b++) {
            const int64_t i = base + b * stride + lane;
            kb[b] = i < per_q ? __hip_atomic_load(src + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
        }
#pragma unroll
        for (int b = 0; b < B; b++) wave_list_offer(kb[b], list, thr, a.k);
    }
    wave_lists_merge(list, thr, a.k, buf);
    if (wave == 0 && lane < a.k) {
        a.out_ids[(int64_t)qi * a.k + lane] = list ? (int32_t)key_index(list) : -1;
        if (a.out_topk_scores) a.out_topk_scores[(int64_t)qi * a.k + lane] = list ? key_score(list, a.smallest) : 0.0f;
    }
    if (threadIdx.x == 0) __hip_atomic_store(&a.tickets[qi], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// -------------------------------------------------- q8, coalesced lanes

// Sum over aligned groups of L lanes (L = 4, 8 or 16) with DPP moves inside
// each 16-lane row; every lane of a group receives the group total.
template <int L>
__device__ __forceinline__ int group_sum(int s) {
    s += __builtin_amdgcn_update_dpp(0, s, 0xB1, 0xf, 0xf, false);  // quad_perm [1,0,3,2]
    s += __builtin_amdgcn_update_dpp(0, s, 0x4E, 0xf, 0xf, false);  // quad_perm [2,3,0,1]
    if (L >= 8) s += __builtin_amdgcn_update_dpp(0, s, 0x141, 0xf, 0xf, false);   // row_half_mirror
    if (L >= 16) s += __builtin_amdgcn_update_dpp(0, s, 0x140, 0xf, 0xf, false);  // row_mirror
    return s;
}

// Buffer resource over `bytes` bytes at p (raw, stride 0): loads at offsets
// at or past `bytes` return zero instead of touching memory.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t byte_buffer(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

template <int CTRL>
__device__ __forceinline__ float dpp_f32(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false));
}

// DPP move of a double: both 32-bit halves with the same pattern.
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double x) {
    const uint64_t b = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, false);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

template <int L>
__device__ __forceinline__ float group_fmax(float m) {
    m = fmaxf(m, dpp_f32<0xB1>(m));
    m = fmaxf(m, dpp_f32<0x4E>(m));
    if (L >= 8) m = fmaxf(m, dpp_f32<0x141>(m));
    if (L >= 16) m = fmaxf(m, dpp_f32<0x140>(m));
    return m;
}

// Exact while every partial sum stays below 2^53 (sums of squared codes).
template <int L>
__device__ __forceinline__ double group_dsum(double s) {
    s += dpp_f64<0xB1>(s);
    s += dpp_f64<0x4E>(s);
    if (L >= 8) s += dpp_f64<0x141>(s);
    if (L >= 16) s += dpp_f64<0x140>(s);
    return s;
}

// Encode the query columns this lane multiplies straight into registers:
// chunk c of lane p covers columns [16*(c*L + p), +16) (zero past d).  The L
// lanes of a group cover every column, so group reductions give the
// whole-query max |q| and sum of squared codes; codes and constants equal
// encode_query_block's.  Whole wave, no LDS, no barrier.
template <int OP, int L, int C>
__device__ __forceinline__ QConst encode_query_lanes(const uint16_t* qrow, int d, int p, v4i* qa, v4i* qb) {
    const __amdgpu_buffer_rsrc_t qr = byte_buffer(qrow, (uint32_t)d * 2u);
    uint16_t hx[C][16];  // raw f16 bits, converted where used
    float m = 0.0f;
#pragma unroll
    for (int c = 0; c < C; c++)
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int col = c * 16 * L + p * 16 + e;
            hx[c][e] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(qr, col * 2, 0, 0);
            m = fmaxf(m, __builtin_fabsf(h2f(hx[c][e])));
        }
    m = group_fmax<L>(m);
    if (OP == OP_DOT) {
        const float qmax = fmaxf(1.0f, m);
#pragma unroll
        for (int c = 0; c < C; c++) {
#pragma unroll
            for (int w = 0; w < 4; w++) {
                int word = 0;
#pragma unroll
                for (int b = 0; b < 4; b++) word |= (code_e8(h2f(hx[c][4 * w + b]), qmax) & 0xFF) << (8 * b);
                qa[c][w] = word;
            }
            qb[c] = qa[c];
        }
        return QConst{qmax, 0.0f, 0.0f, 0.0f};
    }
    const float inv = m == 0.0f ? 0.0f : fdiv_rn(32639.0f, m);
    double ss = 0.0;
#pragma unroll
    for (int c = 0; c < C; c++)
#pragma unroll
        for (int w = 0; w < 4; w++) {
            int hw = 0, lw = 0;
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const int code = m != 0.0f ? code_e16(h2f(hx[c][4 * w + b]), inv) : 0;
                const int l = (int)(int8_t)(code & 0xFF);
                const int h = (code - l) >> 8;
                hw |= (h & 0xFF) << (8 * b);
                lw |= (l & 0xFF) << (8 * b);
                ss += (double)code * (double)code;
            }
            qa[c][w] = hw;
            qb[c][w] = lw;
        }
    ss = group_dsum<L>(ss);
    return e16_consts(m, (long long)ss);
}

// Pitch = 16*L*C bytes.  A wave scores a block of 64 rows per round; lane
// group g (L lanes) owns rows g*L .. g*L+L-1 of the block.  Load (j, c)
// reads row g*L + j, lane p of the group taking bytes [16p + 16Lc, +16), so
// one load instruction reads 64/L whole rows.  The row sum is a DPP group
// sum, and lane g*L + j keeps it: after a round every lane holds the
// accumulator of its own row.  Loads go through a buffer resource clipped to
// the workgroup's rows (no branch per load; rows past n read zero and are
// masked by `valid`).
enum { SCAN_RESERVOIR = 0, SCAN_LISTS = 1, SCAN_BUFFERED = 2 };

template <int OP, int L, int C, int MODE>
__global__ __launch_bounds__(256) void q8_scan_kernel(ScanArgs a) {
    constexpr bool LISTS = MODE == SCAN_LISTS;
    constexpr bool AHEAD = MODE != SCAN_RESERVOIR;  // the next step's loads go out early
    extern __shared__ uint64_t topk_keys[];
    __shared__ ScanTopkLds S;
    __shared__ uint64_t ff_keys[LISTS ? 256 : 1];  // the lists' first fill, 64 keys a wave
    constexpr int PITCH = 16 * L * C;
    constexpr int JS0 = C == 1 ? 16 : (C == 2 ? 8 : 4);  // rows per load step (<= 16 loads)
    constexpr int JS = JS0 < L ? JS0 : L;
    static_assert(L % JS == 0, "load steps must tile the lane group");
    const int qi = blockIdx.y;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int p = lane % L;
    const int g = lane / L;
    const int64_t set_row0 = (int64_t)qi * a.set_stride;
    const int8_t* __restrict__ codes = a.codes + set_row0 * PITCH;
    const float* __restrict__ scales = (const float*)a.scales + set_row0;

    const int64_t wg_row0 = (int64_t)blockIdx.x * a.rounds * 256;
    const int64_t left = a.n - wg_row0;  // > 0: the grid covers n exactly
    const int wg_rows = left < (int64_t)a.rounds * 256 ? (int)left : a.rounds * 256;
    const __amdgpu_buffer_rsrc_t rs = byte_buffer(codes + wg_row0 * PITCH, (uint32_t)wg_rows * PITCH);
    const int lane_off = g * L * PITCH + p * 16;
    // One load step: rows j0 .. j0+JS-1 of every lane group of the wave's
    // block in round r.  On the list and buffered paths the next step's loads are
    // issued as soon as the current step's values are consumed, so they
    // overlap the epilogue and the top-k offer, and the first step's overlap
    // the query encoding.
    v4i v[JS][C];
    auto load_step = [&](int r, int j0) {
        const int vb = (r * 256 + wave * 64) * PITCH + lane_off;
#pragma unroll
        for (int j = 0; j < JS; j++)
#pragma unroll
            for (int c = 0; c < C; c++)
                v[j][c] = __builtin_amdgcn_raw_buffer_load_b128(rs, vb + (j0 + j) * PITCH + c * 16 * L, 0, 2);
    };
    if (AHEAD) load_step(0, 0);

    v4i qa[C], qb[C];
    const QConst kq = encode_query_lanes<OP, L, C>(a.queries + (int64_t)qi * a.d, a.d, p, qa, qb);
    // LISTS: top-k through per-wave register lists (k <= 64, never score mode)
    uint64_t list = 0, thr = 0;
    if (MODE == SCAN_RESERVOIR && !a.out_scores) topk_init(topk_keys, &S.st);

    for (int r = 0; r < a.rounds; r++) {
        const int64_t row = wg_row0 + r * 256 + wave * 64 + lane;
        const bool valid = row < a.n;
        const int64_t crow = valid ? row : a.n - 1;
        const float sc = scales[crow];
        float dn = 0.0f, d2 = 0.0f;
        if (OP == OP_COSINE) dn = a.dnorm[set_row0 + crow];
        if (OP == OP_L2) d2 = a.dd[set_row0 + crow];
        int my_hi = 0, my_lo = 0;
#pragma unroll
        for (int j0 = 0; j0 < L; j0 += JS) {
            // the reservoir path loads each step when it starts (its offer
            // and compaction would otherwise run with a step of loads held)
            if (!AHEAD) load_step(r, j0);
#pragma unroll
            for (int j = 0; j < JS; j++) {
                int s_hi = 0, s_lo = 0;
#pragma unroll
                for (int c = 0; c < C; c++) {
                    s_hi = dot16(v[j][c], qa[c], s_hi);
                    if (OP != OP_DOT) s_lo = dot16(v[j][c], qb[c], s_lo);
                }
                s_hi = group_sum<L>(s_hi);
                if (OP != OP_DOT) s_lo = group_sum<L>(s_lo);
                if (p == j0 + j) {
                    my_hi = s_hi;
                    my_lo = s_lo;
                }
            }
            // the step's values are consumed before the next loads are
            // issued (else the loads would be hoisted and double the
            // registers held)
            asm volatile("" : "+v"(my_hi), "+v"(my_lo));
            asm volatile("" ::: "memory");
            if (!AHEAD) continue;
            // unconditional, so the wait counts stay static: after the last
            // round these loads fall past the buffer and return zeros
            // without touching memory
            if (j0 + JS < L)
                load_step(r, j0 + JS);
            else
                load_step(r + 1, 0);
        }
        float score = 0.0f;
        if (valid) score = q8_epilogue<OP>(my_hi, my_lo, sc, kq, dn, d2);
        if (LISTS) {
            const uint64_t key = valid ? make_key(score, (uint32_t)row, a.smallest) : 0ull;
            // (the lists start empty: the first round fills them by rank,
            // in LDS of its own -- a wave that finishes early may already be
            // merging through topk_keys)
            if (r == 0) wave_list_first_fill(key, list, thr, a.k, ff_keys + wave * 64);
            else wave_list_offer(key, list, thr, a.k);
            continue;
        }
        emit_round(a, score, valid, row, r, qi, topk_keys, &S.st);
    }
    if (LISTS)
        finish_wave_lists(a, list, thr, topk_keys, S, qi);
    else if (MODE == SCAN_BUFFERED)
        finish_buffered(a, topk_keys, qi);
    else if (!a.out_scores)
        finish_topk(a, topk_keys, S, qi);
}

// ------------------------------------------ q8, any pitch (lane = 16 bytes)

// LDS words (int2) a wave of the kernel below trades sums through: 8 loads of
// 64 / nc rows, nc | 1 words each (rows on distinct banks).
__host__ __device__ constexpr int q8_generic_words(int nc) { return 8 * (64 / nc) * (nc | 1); }

// Lane p of a group of pitch/16 lanes takes bytes [16p, +16) of a row, so a
// load instruction reads 64 / (pitch/16) whole rows side by side; the lanes'
// integer sums meet through LDS, one lane adding a row's, a batch of 8 loads at
// a time, and lane i of the wave keeps row i of its 64.  Loads are 8
// instructions ahead, across rounds too.  (A row per lane read 16 bytes out of
// every row per load: two queries over 300,000 rows of 1,000, k = 180, 303 us
// a call against 173.)
template <int OP>
__global__ __launch_bounds__(256) void q8_scan_generic_kernel(ScanArgs a) {
    extern __shared__ uint64_t topk_keys[];
    __shared__ ScanLds S;
    __shared__ int2 sums[4][64];  // a wave's row sums of the round
    constexpr int B = 8;
    const int qi = blockIdx.y;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nc = a.pitch / 16;
    const int rpl = 64 / nc, steps = (64 + rpl - 1) / rpl;  // rows per load, loads per 64 rows
    const int g = lane / nc, p = lane - g * nc;
    const bool act = g < rpl;
    const int64_t set_row0 = (int64_t)qi * a.set_stride;
    const float* __restrict__ scales = (const float*)a.scales + set_row0;
    const int64_t wg_row0 = (int64_t)blockIdx.x * a.rounds * 256;
    const int64_t left = a.n - wg_row0;  // > 0: the grid covers n exactly
    const int wg_rows = left < (int64_t)a.rounds * 256 ? (int)left : a.rounds * 256;
    const __amdgpu_buffer_rsrc_t rs =
        byte_buffer(a.codes + (set_row0 + wg_row0) * a.pitch, (uint32_t)wg_rows * a.pitch);
    // past the buffer, whatever row is added: such loads touch no memory.  (The
    // whole offset is the lanes': the scalar offset has no part in the bounds
    // check.  Unsigned, as the check is: two of them do not wrap.)
    constexpr uint32_t kFar = 0x7ffffff0u;
    const uint32_t voff = act ? (uint32_t)((wave * 64 + g) * a.pitch + p * 16) : kFar;
    v4i w[B], wn[B];
    auto load = [&](v4i (&dw)[B], int r, int s0) {
#pragma unroll
        for (int j = 0; j < B; j++) {
            const bool in = s0 + j < steps;  // the same for the whole wave
            const uint32_t off = in ? (uint32_t)((r * 256 + (s0 + j) * rpl) * a.pitch) : kFar;
            dw[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, voff + off, 0, 2);
        }
    };
    load(w, 0, 0);
    encode_query_block(a.queries + (int64_t)qi * a.d, a.d, a.pitch, OP == OP_DOT ? ENC_E8 : ENC_E16, S.q);
    const QConst kq = S.q.qc;
    const v4i qa = *(const v4i*)((OP == OP_DOT ? S.q.c8 : S.q.hi) + 16 * p);
    const v4i qb = OP == OP_DOT ? qa : *(const v4i*)(S.q.lo + 16 * p);
    const int pp = nc | 1;
    const int H = rpl == 1 ? 8 : (rpl == 2 ? 4 : (rpl <= 4 ? 2 : 1));  // H * 8 * rpl <= 64
    int2* part = (int2*)(topk_keys + a.lds_keys) + wave * q8_generic_words(nc);
    if (!a.out_scores && !a.buffered) topk_init(topk_keys, &S.st);
    for (int r = 0; r < a.rounds; r++) {
        const int64_t row = wg_row0 + (int64_t)r * 256 + wave * 64 + lane;
        const bool valid = row < a.n;
        const int64_t crow = valid ? row : a.n - 1;
        const float sc = scales[crow];
        const float dn = OP == OP_COSINE ? a.dnorm[set_row0 + crow] : 0.0f;
        const float d2 = OP == OP_L2 ? a.dd[set_row0 + crow] : 0.0f;
        for (int s0 = 0; s0 < steps; s0 += B) {
            const bool more = s0 + B < steps;
            load(wn, more ? r : r + 1, more ? s0 + B : 0);
#pragma unroll
            for (int j = 0; j < B; j++) {
                const int hi = dot16(w[j], qa, 0);
                const int lo = OP == OP_DOT ? 0 : dot16(w[j], qb, 0);
                if (act) part[(j * rpl + g) * pp + p] = int2{hi, lo};
            }
#pragma unroll
            for (int j = 0; j < B; j++) w[j] = wn[j];
            // the wave's lanes trade sums: its LDS operations run in order,
            // the empty asm statements keep the compiler to that order
            __builtin_amdgcn_wave_barrier();
            asm volatile("" ::: "memory");
            if (H == 1) {
                for (int br = lane; br < B * rpl; br += 64) {
                    int2 t{0, 0};
#pragma unroll 4
                    for (int c = 0; c < nc; c++) {
                        const int2 e = part[br * pp + c];
                        t.x += e.x, t.y += e.y;
                    }
                    if (s0 * rpl + br < 64) sums[wave][s0 * rpl + br] = t;
                }
            } else {
                // few wide rows: H lanes share a row's words
                const int br = lane / H;
                int2 t{0, 0};
                if (br < B * rpl) {
#pragma unroll 4
                    for (int c = lane & (H - 1); c < nc; c += H) {
                        const int2 e = part[br * pp + c];
                        t.x += e.x, t.y += e.y;
                    }
                }
                for (int off = 1; off < H; off <<= 1) {
                    t.x += __shfl_xor(t.x, off);
                    t.y += __shfl_xor(t.y, off);
                }
                if ((lane & (H - 1)) == 0 && br < B * rpl && s0 * rpl + br < 64) sums[wave][s0 * rpl + br] = t;
            }
            __builtin_amdgcn_wave_barrier();
            asm volatile("" ::: "memory");
        }
        const int2 acc = sums[wave][lane];
        __builtin_amdgcn_wave_barrier();
        asm volatile("" ::: "memory");
        const float score = valid ? q8_epilogue<OP>(acc.x, acc.y, sc, kq, dn, d2) : 0.0f;
        emit_round(a, score, valid, row, r, qi, topk_keys, &S.st);
    }
    if (a.buffered) finish_buffered(a, topk_keys, qi);
    else if (!a.out_scores) finish_topk(a, topk_keys, S, qi);
}

// ------------------------------------------------ q8, any pitch (lane = row)

// A row per lane, 16 bytes of every row per load.  The rows' lines come from
// the caches after their first load; nothing is traded between lanes
// (q8_row_per_lane: where it is the faster one).
template <int OP>
__global__ __launch_bounds__(256) void q8_scan_rows_kernel(ScanArgs a) {
    extern __shared__ uint64_t topk_keys[];
    __shared__ ScanLds S;
    const int qi = blockIdx.y;
    const int64_t set_row0 = (int64_t)qi * a.set_stride;
    const int8_t* __restrict__ codes = a.codes + set_row0 * a.pitch;
    const float* __restrict__ scales = (const float*)a.scales + set_row0;
    encode_query_block(a.queries + (int64_t)qi * a.d, a.d, a.pitch, OP == OP_DOT ? ENC_E8 : ENC_E16, S.q);
    const QConst kq = S.q.qc;
    const int8_t* qa = OP == OP_DOT ? S.q.c8 : S.q.hi;
    const int8_t* qb = S.q.lo;
    const int chunks = a.pitch / 16;
    if (!a.out_scores && !a.buffered) topk_init(topk_keys, &S.st);
    const int64_t wg_row0 = (int64_t)blockIdx.x * a.rounds * 256;
    for (int r = 0; r < a.rounds; r++) {
        const int64_t row = wg_row0 + (int64_t)r * 256 + threadIdx.x;
        const bool valid = row < a.n;
        float score = 0.0f;
        if (valid) {
            const v4i* rp = (const v4i*)(codes + row * a.pitch);
            int s_hi = 0, s_lo = 0;
            for (int c = 0; c < chunks; c++) {
                const v4i v = rp[c];
                s_hi = dot16(v, *(const v4i*)(qa + c * 16), s_hi);
                if (OP != OP_DOT) s_lo = dot16(v, *(const v4i*)(qb + c * 16), s_lo);
            }
            const float dn = OP == OP_COSINE ? a.dnorm[set_row0 + row] : 0.0f;
            const float d2 = OP == OP_L2 ? a.dd[set_row0 + row] : 0.0f;
            score = q8_epilogue<OP>(s_hi, s_lo, scales[row], kq, dn, d2);
        }
        emit_round(a, score, valid, row, r, qi, topk_keys, &S.st);
    }
    if (a.buffered) finish_buffered(a, topk_keys, qi);
    else if (!a.out_scores) finish_topk(a, topk_keys, S, qi);
}

// ------------------------------------------------------- q4, lane = block

// Lane p of a group of nb lanes takes block p of a row, so a load instruction
// reads 64 / nb whole rows side by side (16 bytes a lane, the block's f16 scale
// beside it) and the lane's 32 query codes stay in registers.  The contract's
// fma chain runs over a row's blocks in order, so the block sums go through
// LDS as (scale, sum) pairs and lane i of the wave folds row i of its 64 (pair
// pitch nb | 1: 64 rows on distinct banks).  Loads are 8 instructions ahead,
// across rounds too.  The read of the rows bounds it: one query against
// 1,048,576 x 384 rows took 167 us with a row per lane (16 bytes out of every
// 192 per load), 65 this way with the selection (226 MB: 46 us at the copy
// rate).
template <int OP>
__global__ __launch_bounds__(256) void q4_scan_kernel(ScanArgs a) {
    extern __shared__ uint64_t topk_keys[];
    __shared__ ScanLds S;
    constexpr int B = 8;
    const int qi = blockIdx.y;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nb = a.nb;
    const int rpl = 64 / nb, steps = (64 + rpl - 1) / rpl;  // rows per load, loads per 64 rows
    const int g = lane / nb, p = lane - g * nb;
    const bool act = g < rpl;
    const int64_t set_row0 = (int64_t)qi * a.set_stride;
    const int64_t wg_row0 = (int64_t)blockIdx.x * a.rounds * 256;
    const int64_t left = a.n - wg_row0;  // > 0: the grid covers n exactly
    const int wg_rows = left < (int64_t)a.rounds * 256 ? (int)left : a.rounds * 256;
    const __amdgpu_buffer_rsrc_t rs =
        byte_buffer((const uint8_t*)a.codes + (set_row0 + wg_row0) * a.pitch, (uint32_t)wg_rows * a.pitch);
    const __amdgpu_buffer_rsrc_t ss =
        byte_buffer((const uint16_t*)a.scales + (set_row0 + wg_row0) * nb, (uint32_t)wg_rows * nb * 2);
    // past every buffer, whatever row is added: such loads touch no memory
    // (the whole offset is the lanes', as above)
    constexpr uint32_t kFar = 0x7ffffff0u;
    const uint32_t voff = act ? (uint32_t)((wave * 64 + g) * a.pitch + p * 16) : kFar;
    const uint32_t soff = act ? (uint32_t)(((wave * 64 + g) * nb + p) * 2) : kFar;
    v4i w[B], wn[B];
    uint16_t sc[B], scn[B];
    auto load = [&](v4i (&dw)[B], uint16_t (&ds)[B], int r, int s0) {
#pragma unroll
        for (int j = 0; j < B; j++) {
            const int row = r * 256 + (s0 + j) * rpl;
            const bool in = s0 + j < steps;  // the same for the whole wave
            dw[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, voff + (in ? (uint32_t)(row * a.pitch) : kFar), 0, 2);
            ds[j] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(ss, soff + (in ? (uint32_t)(row * nb * 2) : kFar), 0, 2);
        }
    };
    load(w, sc, 0, 0);
    encode_query_block(a.queries + (int64_t)qi * a.d, a.d, a.d, ENC_E16_Q4, S.q);
    const QConst kq = S.q.qc;
    int qh[8], ql[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        qh[j] = ((const int*)S.q.hi)[8 * p + j];
        ql[j] = ((const int*)S.q.lo)[8 * p + j];
    }
    const int pp = nb | 1;
    float2* pairs = (float2*)(topk_keys + a.lds_keys) + wave * 64 * pp;
    if (!a.out_scores && !a.buffered) topk_init(topk_keys, &S.st);
    for (int r = 0; r < a.rounds; r++) {
        const int64_t row = wg_row0 + (int64_t)r * 256 + wave * 64 + lane;
        const bool valid = row < a.n;
        const int64_t crow = set_row0 + (valid ? row : a.n - 1);
        const float dn = OP == OP_COSINE ? a.dnorm[crow] : 0.0f;
        const float d2 = OP == OP_L2 ? a.dd[crow] : 0.0f;
        for (int s0 = 0; s0 < steps; s0 += B) {
            const bool more = s0 + B < steps;
            load(wn, scn, more ? r : r + 1, more ? s0 + B : 0);
#pragma unroll
            for (int j = 0; j < B; j++) {
                const int lr = (s0 + j) * rpl + g;  // row of the wave's 64
                const float acc = (float)q4_block_acc(w[j], qh, ql);
                if (act && lr < 64) pairs[lr * pp + p] = float2{h2f(sc[j]), acc};
            }
#pragma unroll
            for (int j = 0; j < B; j++) w[j] = wn[j], sc[j] = scn[j];
        }
        // the wave's lanes trade pairs: its LDS operations run in order, the
        // empty asm statements keep the compiler to that order
        __builtin_amdgcn_wave_barrier();
        asm volatile("" ::: "memory");
        float dotf = 0.0f;
#pragma unroll 4
        for (int b = 0; b < nb; b++) {
            const float2 e = pairs[lane * pp + b];
            dotf = __fmaf_rn(e.x, e.y, dotf);
        }
        __builtin_amdgcn_wave_barrier();
        asm volatile("" ::: "memory");
        const float score = valid ? q4_finish<OP>(dotf, kq, dn, d2) : 0.0f;
        emit_round(a, score, valid, row, r, qi, topk_keys, &S.st);
    }
    if (a.buffered) finish_buffered(a, topk_keys, qi);
    else if (!a.out_scores) finish_topk(a, topk_keys, S, qi);
}

// A row per lane: no pairs go through LDS, each lane runs its row's chain
// (q4_row_per_lane: where it is the faster one).
template <int OP>
__global__ __launch_bounds__(256) void q4_scan_rows_kernel(ScanArgs a) {
    extern __shared__ uint64_t topk_keys[];
    __shared__ ScanLds S;
    const int qi = blockIdx.y;
    const int64_t set_row0 = (int64_t)qi * a.set_stride;
    const uint8_t* __restrict__ packed = (const uint8_t*)a.codes + set_row0 * a.pitch;
    const uint16_t* __restrict__ scales = (const uint16_t*)a.scales + set_row0 * a.nb;
    encode_query_block(a.queries + (int64_t)qi * a.d, a.d, a.d, ENC_E16_Q4, S.q);
    const QConst kq = S.q.qc;
    if (!a.out_scores && !a.buffered) topk_init(topk_keys, &S.st);
    const int64_t wg_row0 = (int64_t)blockIdx.x * a.rounds * 256;
    for (int r = 0; r < a.rounds; r++) {
        const int64_t row = wg_row0 + (int64_t)r * 256 + threadIdx.x;
        const bool valid = row < a.n;
        float score = 0.0f;
        if (valid) {
            const float dotf = q4_row_dotf(packed + row * a.pitch, scales + row * a.nb, a.nb, (const int*)S.q.hi,
                                           (const int*)S.q.lo);
            const float dn = OP == OP_COSINE ? a.dnorm[set_row0 + row] : 0.0f;
            const float d2 = OP == OP_L2 ? a.dd[set_row0 + row] : 0.0f;
            score = q4_finish<OP>(dotf, kq, dn, d2);
        }
        emit_round(a, score, valid, row, r, qi, topk_keys, &S.st);
    }
    if (a.buffered) finish_buffered(a, topk_keys, qi);
    else if (!a.out_scores) finish_topk(a, topk_keys, S, qi);
}

// ------------------------------------------------ exact accumulator rescore

// One workgroup per query: re-encode the query and recompute the q8
// integer accumulator of each selected row (E8 for dot, E16 hi/lo combined
// for the others), written as int64.
__global__ __launch_bounds__(256) void q8_rescore_acc_kernel(const int8_t* __restrict__ codes, int pitch,
                                                             int64_t set_stride, int64_t n, int d,
                                                             const uint16_t* __restrict__ queries,
                                                             const int32_t* __restrict__ ids, int k, int e16,
                                                             int64_t* __restrict__ out) {
    __shared__ QueryLds L;
    const int qi = blockIdx.x;
    encode_query_block(queries + (int64_t)qi * d, d, pitch, e16 ? ENC_E16 : ENC_E8, L);
    for (int i = threadIdx.x; i < k; i += blockDim.x) {
        const int64_t row = ids[(int64_t)qi * k + i];
        int64_t acc = 0;
        if (row >= 0 && row < n) {
            const int8_t* rp = codes + ((int64_t)qi * set_stride + row) * pitch;
            for (int c = 0; c < pitch; c++)
                acc += (int64_t)rp[c] * (e16 ? 256 * (int64_t)L.hi[c] + L.lo[c] : (int64_t)L.c8[c]);
        }
        out[(int64_t)qi * k + i] = acc;
    }
}

// ----------------------------------------------------------------- hosts

hipError_t launch_query_encode(const uint16_t* q, int nq, int d, int pitch, int e16, int8_t* c8,
                               int8_t* hi, int8_t* lo, QConst* qc, uint64_t* tau, int* bcnt, hipStream_t s) {
    hipLaunchKernelGGL(query_encode_kernel, dim3(nq), dim3(256), 0, s, q, d, pitch, e16, c8, hi, lo, qc, tau, bcnt);
    return hipGetLastError();
}

hipError_t launch_query_encode_shadow(const uint16_t* q, int nq, int d, int spitch, int op, const ShadowInfo* info,
                                      int8_t* c8, int8_t* hi, int8_t* lo, QConst* qc, float* qb, uint64_t* tau,
                                      int* bcnt, hipStream_t s) {
    if (d % 32 != 0 || d > kMaxQueryDim || spitch < d) return hipErrorInvalidValue;
    hipLaunchKernelGGL(query_encode_shadow_kernel, dim3(nq), dim3(256), 0, s, q, d, spitch, op, info, c8, hi, lo, qc,
                       qb, tau, bcnt);
    return hipGetLastError();
}

bool q8_scan_coalesced(int pitch) {
    const int chunks = pitch / 16;
    return pitch % 16 == 0 && (chunks == 4 || chunks == 8 || chunks == 12 || chunks == 16 || chunks == 24 ||
                               chunks == 32 || chunks == 48 || chunks == 64);
}

// A row per lane, or the pieces of a row side by side over the lanes.  A row
// per lane reads 16 bytes out of every row at a time: fine while the rows stay
// in the caches between its loads, and it trades no sums between lanes.  Whole
// calls, us, row per lane / pieces, dot, k = 8, queries x rows:
//   q8, d           1 x 30,000    7 x 150,000   1 x 500,000   7 x 500,000   3 x 1,500,000
//    40 (48 bytes)  11.0 / 13.3   27.1 / 35.4   16.3 / 23.4   44.7 / 54.4   47.7 / 62.6
//   100             11.8 / 13.5   35.5 / 35.9   23.2 / 23.7  105.8 / 77.7  126.1 / 66.6
//   200             12.8 / 14.7   47.0 / 49.5   29.6 / 29.4  111.6 / 116.7 158.1 / 111.7
//   400             14.2 / 18.8   76.6 / 81.8   44.1 / 44.5  160.8 / 221.1
//   600             16.1 / 25.4  114.7 / 145.3  79.0 / 72.1  311.4 / 403.9
//   1,000           21.6 / 28.6  177.5 / 176.4  (7 x 300,000, k = 5: 372 / 284)
//   q4, d
//    64             11.2 / 13.2   21.5 / 32.7   16.1 / 22.1   33.1 / 50.2   36.0 / 57.0
//   160             12.0 / 13.9   30.0 / 36.6   20.8 / 24.0   60.7 / 67.7   64.5 / 75.4
//   256             13.1 / 14.2   40.7 / 40.1   25.9 / 25.8   99.2 / 90.8  104.8 / 95.7
//   384             13.9 / 16.2   57.8 / 63.5   34.7 / 36.2  142.9 / 156.0 177.6 / 158.0
//   512             16.4 / 17.4   72.7 / 63.5   41.5 / 39.4  193.9 / 160.6 258.9 / 217.7
//   1,024           22.0 / 23.6  135.1 / 113.6  84.5 / 64.0  434.9 / 295.6
constexpr int64_t kMB = 1 << 20;

static bool q8_row_per_lane(const ScanArgs& a, int64_t nq) {
    const int chunks = a.pitch / 16;
    if (chunks <= 3) return true;
    const int64_t one = a.n * a.pitch, all = one * nq, rows = a.set_stride ? all : one;  // bytes: read, and distinct
    // (33 to 52 pieces: a load takes one row and leaves up to half the lanes idle)
    if (chunks > 32 && chunks <= 52 && nq > 1 && !a.set_stride) return true;
    return rows < (chunks > 52 ? 160 : 256) * kMB && (chunks > 8 || all < 80 * kMB);
}

static bool q4_row_per_lane(const ScanArgs& a, int64_t nq) {
    if (a.nb <= 5) return true;
    const int64_t one = a.n * a.pitch, all = one * nq, rows = a.set_stride ? all : one;
    // (8 blocks: every row starts on the same few cache sets, as 16 and 32 do)
    return a.nb <= 12 && a.nb != 8 ? rows < 128 * kMB : all < 32 * kMB;
}

template <int OP>
static hipError_t launch_q8_op(const ScanArgs& a, dim3 grid, size_t lds, hipStream_t s) {
    const int chunks = a.pitch / 16;
    // the list path's merges use 64 LDS keys per wave
    if (a.wave_lists && !a.out_scores && lds < 256 * sizeof(uint64_t)) return hipErrorInvalidValue;
#define MANTA_Q8(LL, CC)                                                                           \
    if (chunks == (LL) * (CC)) {                                                                   \
        if (a.wave_lists && !a.out_scores)                                                                    \
            hipLaunchKernelGGL((q8_scan_kernel<OP, LL, CC, SCAN_LISTS>), grid, dim3(256), lds, s, a);        \
        else if (a.buffered && !a.out_scores)                                                                 \
            hipLaunchKernelGGL((q8_scan_kernel<OP, LL, CC, SCAN_BUFFERED>), grid, dim3(256), lds, s, a);     \
        else                                                                                                  \
            hipLaunchKernelGGL((q8_scan_kernel<OP, LL, CC, SCAN_RESERVOIR>), grid, dim3(256), lds, s, a);    \
        return hipGetLastError();                                                                             \
    }
    MANTA_Q8(4, 1)    // d <= 64
    MANTA_Q8(8, 1)    // 128
    MANTA_Q8(4, 3)    // 192
    MANTA_Q8(16, 1)   // 256
    MANTA_Q8(8, 3)    // 384
    MANTA_Q8(16, 2)   // 512
    MANTA_Q8(16, 3)   // 768
    MANTA_Q8(16, 4)   // 1024
#undef MANTA_Q8
    if (chunks < 1 || chunks > 64 || a.pitch != 16 * chunks || lds < (size_t)a.lds_keys * 8) return hipErrorInvalidValue;
    if (q8_row_per_lane(a, grid.y)) {
        hipLaunchKernelGGL((q8_scan_rows_kernel<OP>), grid, dim3(256), lds, s, a);
        return hipGetLastError();
    }
    const size_t all = (size_t)a.lds_keys * 8 + (size_t)4 * q8_generic_words(chunks) * sizeof(int2);
    hipLaunchKernelGGL((q8_scan_generic_kernel<OP>), grid, dim3(256), all, s, a);
    return hipGetLastError();
}

hipError_t launch_q8_scan(int op, const ScanArgs& a, dim3 grid, size_t lds, hipStream_t s) {
    switch (op) {
        case OP_DOT: return launch_q8_op<OP_DOT>(a, grid, lds, s);
        case OP_DOT16: return launch_q8_op<OP_DOT16>(a, grid, lds, s);
        case OP_COSINE: return launch_q8_op<OP_COSINE>(a, grid, lds, s);
        default: return launch_q8_op<OP_L2>(a, grid, lds, s);
    }
}

template <int OP>
static hipError_t launch_q4_op(const ScanArgs& a, dim3 grid, size_t lds, hipStream_t s) {
    if (q4_row_per_lane(a, grid.y)) {
        hipLaunchKernelGGL((q4_scan_rows_kernel<OP>), grid, dim3(256), lds, s, a);
        return hipGetLastError();
    }
    const size_t all = (size_t)a.lds_keys * 8 + (size_t)4 * 64 * (a.nb | 1) * sizeof(float2);  // + (scale, sum) pairs
    hipLaunchKernelGGL((q4_scan_kernel<OP>), grid, dim3(256), all, s, a);
    return hipGetLastError();
}

hipError_t launch_q4_scan(int op, const ScanArgs& a, dim3 grid, size_t lds, hipStream_t s) {
    if (a.nb < 1 || a.nb > 32 || a.pitch != 16 * a.nb || lds < (size_t)a.lds_keys * 8) return hipErrorInvalidValue;
    switch (op) {
        case OP_DOT: return launch_q4_op<OP_DOT>(a, grid, lds, s);
        case OP_COSINE: return launch_q4_op<OP_COSINE>(a, grid, lds, s);
        default: return launch_q4_op<OP_L2>(a, grid, lds, s);
    }
}

hipError_t launch_q8_rescore(const int8_t* codes, int pitch, int64_t set_stride, int64_t n, int d,
                             const uint16_t* queries, const int32_t* ids, int k, int nq, int e16,
                             int64_t* out, hipStream_t s) {
    hipLaunchKernelGGL(q8_rescore_acc_kernel, dim3(nq), dim3(256), 0, s, codes, pitch, set_stride, n, d,
                       queries, ids, k, e16, out);
    return hipGetLastError();
}

}  // namespace manta
