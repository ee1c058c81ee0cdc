// kernels_enc16.hip -- the encoder forward with its weight products on the
// f16 matrix cores (d and h multiples of 128): q8 weights widened exactly to
// f16 [N][K], their column scales applied after the f32 accumulation, the
// left operands rounded to f16 by the steps that produce them.  Everything
// else is f32 (f64 where the reference uses it: the softmax exponentials and
// sum, the layernorm's reciprocal square root, the norm of a row).
//
//   enc_prep_kernel       all six weights to f16 [N][K], one launch
//   enc_gather16_kernel   token rows code * scale, rounded to f16
//   enc_gemm16_kernel     a weight product with its epilogue: f32 output (q, k
//                         and v in one launch), gelu and f16 output, or
//                         residual add + layernorm (+ row norm and column sums)
//   enc_attention_kernel  softmax(q k^T) v of one sequence's 64 rows
//   enc_pool_slabs_kernel masked mean over a sequence, f16 output
#include "device_common.hpp"
#include "kernels.hpp"

#pragma clang fp contract(off)

namespace manta {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));

// Direct-to-LDS load (gfx950): each lane's 16 bytes land at M0 + 16*lane.
__device__ __forceinline__ void lds_load16(const void* src, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds) : "memory", "m0");
}

// vmcnt(J*L) + barrier while at least J chunks were issued after the current
// one, else the next smaller J (a smaller count only waits longer).
template <int L, int J>
__device__ __forceinline__ void wait_barrier(int after) {
    if constexpr (J <= 0) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    } else {
        if (after >= J)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(J * L) : "memory");
        else
            wait_barrier<L, J - 1>(after);
    }
}

// geluTensor as v / (1 + exp(-2u)), u = 0.7978845608 (v + 0.044715 v^3): 0.5 (1 +
// tanh u) is that quotient, and without the sum 1 + tanh there is nothing to
// cancel for negative v: the relative error over -4 < v < 0 is below 1e-6
// where 1 + tanhf's reaches 1.5e-3, and the same 2e-7 for positive v.  The
// constants carry the 2 and log2(e).
__device__ __forceinline__ float gelu_sigmoid(float v) {
    const float w = __fmaf_rn(v * v, -0.10294324f, -2.3022082f);
    return v * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(v * w));
}

// Sums of 16 per-lane values over the 32 lanes of each half wave: lane l32
// gets the total of value l32 % 16 (each exchange halves the values a lane
// still holds).
template <typename F>
__device__ __forceinline__ F half_sums(F (&s)[16], int l32) {
#pragma unroll
    for (int step = 8; step >= 1; step >>= 1)
#pragma unroll
        for (int i = 0; i < step; i++) {
            const bool up = (l32 & step) != 0;
            const F a = s[i], b = s[i + step];
            s[i] = (up ? b : a) + __shfl_xor(up ? a : b, step);
        }
    return s[0] + __shfl_xor(s[0], 16);
}

// Maximum and sum over each 16-lane row by DPP moves (quad xor 1, xor 2, half
// mirror, mirror): every lane gets its row's.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, false);
}
template <int CTRL>
__device__ __forceinline__ float dpp_move(float x) {
    return __uint_as_float(dpp_u32<CTRL>(__float_as_uint(x)));
}
template <int CTRL>
__device__ __forceinline__ double dpp_move(double x) {
    const uint64_t b = __builtin_bit_cast(uint64_t, x);
    return __builtin_bit_cast(double, ((uint64_t)dpp_u32<CTRL>((uint32_t)(b >> 32)) << 32) | dpp_u32<CTRL>((uint32_t)b));
}
__device__ __forceinline__ float row16_max(float m) {
    m = fmaxf(m, dpp_move<0xB1>(m));
    m = fmaxf(m, dpp_move<0x4E>(m));
    m = fmaxf(m, dpp_move<0x141>(m));
    return fmaxf(m, dpp_move<0x140>(m));
}
__device__ __forceinline__ double row16_sum(double s) {
    s += dpp_move<0xB1>(s);
    s += dpp_move<0x4E>(s);
    s += dpp_move<0x141>(s);
    return s + dpp_move<0x140>(s);
}

}  // namespace

// ------------------------------------------------------- weights and tokens

// Wt[n][k] = f16(W[k][n]) of the six weights: grid.x counts the 32 x 32 tiles
// of all of them.
__global__ __launch_bounds__(256) void enc_prep_kernel(EncPrepArgs a) {
    __shared__ uint16_t t[32][33];
    int i = 0;
    while (i < 5 && (int)blockIdx.x >= a.first[i + 1]) i++;
    const int K = a.K[i], N = a.N[i], tile = (int)blockIdx.x - a.first[i];
    const int k0 = tile / (N / 32) * 32, n0 = tile % (N / 32) * 32;
    const int8_t* src = a.codes[i];
    uint16_t* dst = a.wt[i];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int r = ty; r < 32; r += 8) t[r][tx] = f2h((float)src[(int64_t)(k0 + r) * N + n0 + tx]);
    __syncthreads();
    for (int r = ty; r < 32; r += 8) dst[(int64_t)(n0 + r) * K + k0 + tx] = t[tx][r];
}

hipError_t launch_enc_prep(EncPrepArgs& a, hipStream_t s) {
    int n = 0;
    for (int i = 0; i < 6; i++) {
        if (a.K[i] % 32 || a.N[i] % 32) return hipErrorInvalidValue;
        a.first[i] = n;
        n += (a.K[i] / 32) * (a.N[i] / 32);
    }
    hipLaunchKernelGGL(enc_prep_kernel, dim3((unsigned)n), dim3(256), 0, s, a);
    return hipGetLastError();
}

// x16[i][c] = f16(codes[tok[i]][c] * scale[tok[i]]), 8 columns a thread; an id
// out of range is recorded in err (report_gather_error: the first position and
// its id) and its row is zero.
__global__ __launch_bounds__(256) void enc_gather16_kernel(const int32_t* __restrict__ tok, int64_t rows,
                                                           const int8_t* __restrict__ codes,
                                                           const float* __restrict__ scales, int64_t vocab, int d,
                                                           uint16_t* __restrict__ x16, unsigned long long* err) {
    const int per = d / 8;
    const int64_t total = rows * per;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int64_t r = i / per;
        const int c = (int)(i - r * per) * 8;
        const int id = tok[r];
        const bool ok = id >= 0 && (int64_t)id < vocab;
        if (!ok && c == 0) report_gather_error(err, r, id);
        const uint2 w = ok ? *(const uint2*)(codes + (int64_t)id * d + c) : uint2{0, 0};
        const float sc = ok ? scales[id] : 0.0f;
        h8 o;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const uint32_t word = e < 4 ? w.x : w.y;
            o[e] = (_Float16)fmul_rn((float)((int)(word << (24 - 8 * (e & 3))) >> 24), sc);
        }
        *(h8*)(x16 + r * d + c) = o;
    }
}

hipError_t launch_enc_gather16(const int32_t* tok, int64_t rows, const int8_t* codes, const float* scales,
                               int64_t vocab, int d, uint16_t* x16, unsigned long long* err, hipStream_t s) {
    if (d % 8 != 0 || ((uintptr_t)codes & 7) != 0) return hipErrorInvalidValue;
    const int64_t g = (rows * (d / 8) + 255) / 256;
    hipLaunchKernelGGL(enc_gather16_kernel, dim3((unsigned)(g < 16384 ? g : 16384)), dim3(256), 0, s, tok, rows, codes,
                       scales, vocab, d, x16, err);
    return hipGetLastError();
}

// ---------------------------------------------------------- weight products

// out = A [M][K] x Bt^T ([N][K]), tiles of MT rows x NT columns by 8 waves:
// MT = 256 four row groups of 64 x two column groups, MT = 64 two of 32 x
// four.  K moves in chunks of 32 through a ring of LDS stages filled by
// direct-to-LDS loads; each 64-byte LDS row stores its 16-byte column c at
// c ^ ((row >> 2) & 3), so the 32 lanes reading one column of 32 rows spread
// over the banks.  Rows past M read the last row and are not stored.  The
// 8 row tiles dealt to the 8 XCDs side by side take their column tiles one
// after the other, so a row tile is read into one L2 only.
//
// Measured (65,536 rows, d 384, h 1536; the previous kernels in parentheses,
// separate layernorm, normalize and pool launches included): q, k, v 97 us
// (218), attn_o + layernorm 65 (171), ffn_up + gelu 126 (297), projection +
// layernorm + norm + pool 146 (396).
//
// The layernorm epilogues need whole rows (NT = N): the residual is added in
// registers, a row's sums go over its lanes by halving exchanges and over the
// column groups through LDS (f32 sums of the values, then of the squared
// deviations; f64 for the row norm), so the product, its sum with the
// residual and the normalized rows never travel through HBM.  What it costs:
// a wave of the 256 x 384 tile holds 192 accumulators, and the row sums beside
// them spill (the compiler's report, bytes a lane and registers: layernorm 300
// and 76, with the token rows as residual 104 and 25, with norm and sums 316 and
// 84; the other tiles none).
template <int MT, int NT>
struct EncTile {
    static constexpr int RG = MT == 256 ? 4 : 2, CG = 8 / RG;
    static constexpr int RB = MT / (32 * RG), CB = NT / (32 * CG);
    static constexpr int AST = MT * 64, BST = NT * 64, STAGE = AST + BST;
    static constexpr int NST = MT == 256 ? 3 : 4;
    static constexpr int ASEG = MT / 16, BSEG = NT / 128;  // 1 KB loads: A in all, B per wave
    static constexpr int LPW = (ASEG >= 8 ? ASEG / 8 : 0) + BSEG;  // at least this many per wave and chunk
    static constexpr size_t LDS = (size_t)NST * STAGE;
};

// TOK: the residual is the q8 token rows (else a.res).
template <int MT, int NT, int EPI, bool TOK>
__global__ __launch_bounds__(512) void enc_gemm16_kernel(EncGemmArgs a) {
    typedef EncTile<MT, NT> TL;
    constexpr int RB = TL::RB, CB = TL::CB, NST = TL::NST;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int rg = wave % TL::RG, cg = wave / TL::RG;
    const int ctn = a.N / NT;
    const unsigned grp = blockIdx.x / (8u * ctn), rem = blockIdx.x - grp * 8u * ctn;
    const int64_t rt = (int64_t)grp * 8 + (rem & 7);
    const int n0 = (int)(rem >> 3) * NT;
    const int64_t m0 = rt * MT;
    if (m0 >= a.M) return;
    const int K = a.K;
    // the token rows a first block adds as its residual: row and scale (0 for
    // a bad id) of each tile row, for the epilogue
    constexpr bool LN = EPI == ENC_EPI_LN || EPI == ENC_EPI_LN_POOL;
    __shared__ __attribute__((aligned(16))) int tok_id[TOK ? MT : 4];
    __shared__ __attribute__((aligned(16))) float tok_sc[TOK ? MT : 4];
    __shared__ __attribute__((aligned(16))) float rowv[LN ? MT : 4];  // a value per row
    __shared__ float part[LN ? TL::CG * MT : 4];                      // row sums of the column groups
    __shared__ double dpart[EPI == ENC_EPI_LN_POOL ? TL::CG * MT : 2];
    if (TOK && tid < MT) {
        const int id = a.tok[m0 + tid < a.M ? m0 + tid : a.M - 1];
        const bool ok = id >= 0 && (int64_t)id < a.vocab;
        tok_id[tid] = ok ? id : 0;
        tok_sc[tid] = ok ? a.res_scales[id] : 0.0f;
    }

    constexpr int AW = TL::ASEG >= 8 ? TL::ASEG / 8 : 1;
    const uint8_t* asrc[AW];
    const bool has_a = TL::ASEG >= 8 || wave < TL::ASEG;
#pragma unroll
    for (int u = 0; u < AW; u++) {
        const int r = 16 * ((AW * wave + u) % TL::ASEG) + (lane >> 2);
        const int64_t row = m0 + r < a.M ? m0 + r : a.M - 1;
        asrc[u] = (const uint8_t*)a.A + row * K * 2 + ((lane & 3) ^ ((r >> 2) & 3)) * 16;
    }
    const uint8_t* bsrc[TL::BSEG];
#pragma unroll
    for (int u = 0; u < TL::BSEG; u++) {
        const int n = 16 * (TL::BSEG * wave + u) + (lane >> 2);
        bsrc[u] = (const uint8_t*)a.Bt + (int64_t)(n0 + n) * K * 2 + ((lane & 3) ^ ((n >> 2) & 3)) * 16;
    }
    const uint32_t base = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)smem);
    auto issue = [&](int kc, int st) {
        const uint32_t sa = __builtin_amdgcn_readfirstlane(base + st * TL::STAGE + wave * AW * 1024);
        if (has_a) {
#pragma unroll
            for (int u = 0; u < AW; u++) lds_load16(asrc[u] + kc * 64, sa + u * 1024);
        }
        const uint32_t sb = __builtin_amdgcn_readfirstlane(base + st * TL::STAGE + TL::AST + wave * TL::BSEG * 1024);
#pragma unroll
        for (int u = 0; u < TL::BSEG; u++) lds_load16(bsrc[u] + kc * 64, sb + u * 1024);
    };
    const int nk = K / 32;
#pragma unroll
    for (int st = 0; st < NST - 1; st++)
        if (st < nk) issue(st, st);

    f16v acc[RB][CB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int cb = 0; cb < CB; cb++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[rb][cb][r] = 0.0f;

    const int l32 = lane & 31, hf = lane >> 5;
    int st = 0;
    for (int kc = 0; kc < nk; kc++, st = st == NST - 1 ? 0 : st + 1) {
        wait_barrier<TL::LPW, NST - 2>(nk - 1 - kc);
        if (kc + NST - 1 < nk) issue(kc + NST - 1, st == 0 ? NST - 1 : st - 1);
        const uint8_t* As = smem + st * TL::STAGE;
        const uint8_t* Bs = As + TL::AST;
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            const int c = ks * 2 + hf;
            h8 av[RB];
#pragma unroll
            for (int rb = 0; rb < RB; rb++) {
                const int r = 32 * (RB * rg + rb) + l32;
                av[rb] = *(const h8*)(As + r * 64 + ((c ^ ((r >> 2) & 3)) * 16));
            }
#pragma unroll
            for (int cb = 0; cb < CB; cb++) {
                const int n = 32 * (CB * cg + cb) + l32;
                const h8 bv = *(const h8*)(Bs + n * 64 + ((c ^ ((n >> 2) & 3)) * 16));
#pragma unroll
                for (int rb = 0; rb < RB; rb++)
                    acc[rb][cb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[rb], bv, acc[rb][cb], 0, 0, 0);
            }
        }
    }

    // Output element (rb, cb, r): row 32*(RB*rg + rb) + 8*(r/4) + 4*(lane/32) +
    // r%4 of the tile, column 32*(CB*cg + cb) + lane%32.
    const int mat = EPI == ENC_EPI_F32 ? n0 / a.D : 0;  // the output matrix of this column tile
    const int nb = n0 - mat * a.D + 32 * CB * cg + l32;
    const int lrow = 32 * RB * rg + 4 * hf;                                // + 32 rb + 8 (r / 4) + r % 4
    const int mlim = a.M - m0 < MT ? (int)(a.M - m0) : MT;                 // rows of this tile
    auto row_of = [&](int rb, int r) { return lrow + 32 * rb + 8 * (r >> 2) + (r & 3); };
    {
        const float* cs = a.colscale[mat];
#pragma unroll
        for (int cb = 0; cb < CB; cb++) {
            const float c = cs[nb + 32 * cb];
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[rb][cb][r] = fmul_rn(acc[rb][cb][r], c);
        }
    }
    if (EPI == ENC_EPI_F32) {
        float* y = a.Y + ((int64_t)mat * a.M + m0) * a.D + nb;
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = row_of(rb, r);
                if (m >= mlim) continue;
#pragma unroll
                for (int cb = 0; cb < CB; cb++) y[m * a.D + 32 * cb] = acc[rb][cb][r];
            }
        return;
    }
    if (EPI == ENC_EPI_GELU16) {
        uint16_t* y = a.Y16 + m0 * a.N + nb;
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = row_of(rb, r);
                if (m >= mlim) continue;
#pragma unroll
                for (int cb = 0; cb < CB; cb++) y[m * a.N + 32 * cb] = f2h(gelu_sigmoid(acc[rb][cb][r]));
            }
        return;
    }
    // Rows leave (and f32 residuals arrive) 8 at a time through two LDS
    // buffers of the wave's own, where the stages were, so that global traffic
    // moves 16 bytes a lane: the accumulators' own layout is 4 bytes a lane,
    // four times the instructions (attn_o's product of 65,536 rows: 116 -> 65
    // us; the other epilogues, stores alone, are no faster this way).  Piece (rb, g) holds rows 32 rb + 8 g + 0..7
    // of the wave's; a row's pitch puts the two half waves on different banks.
    constexpr int WCOL = 32 * CB, WP = WCOL + 8;
    constexpr int WB = 8 * WP * 4;
    static_assert((size_t)16 * WB <= TL::LDS, "two buffers a wave fit the stages");
    float* wbuf = (float*)(smem + wave * 2 * WB);
    const uint32_t wlds = __builtin_amdgcn_readfirstlane(base + wave * 2 * WB);
    const int wrow = 32 * RB * rg;  // the wave's first row of the tile
    const int ncol = n0 - mat * a.D + WCOL * cg;
    auto wave_fence = [] {
        __builtin_amdgcn_wave_barrier();
        asm volatile("" ::: "memory");
    };
    // piece p of the accumulators to fn(row of the tile, column of the matrix, four values)
    auto rows_out = [&](auto fn) {
#pragma unroll
        for (int p = 0; p < 4 * RB; p++) {
            float* buf = wbuf + (p & 1) * (WB / 4);
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int cb = 0; cb < CB; cb++) buf[(4 * hf + e) * WP + 32 * cb + l32] = acc[p >> 2][cb][4 * (p & 3) + e];
            wave_fence();
#pragma unroll
            for (int j = 0; j < CB; j++) {
                const int i = lane + 64 * j, r = i / (8 * CB), c = (i - r * 8 * CB) * 4;
                const int m = wrow + 8 * p + r;
                if (m < mlim) fn(m, ncol + c, *(const float4*)(buf + r * WP + c));
            }
            wave_fence();
        }
    };
    __syncthreads();  // every wave is done with the stage buffers
    auto row4 = [&](int rb, int g) { return *(const float4*)(rowv + lrow + 32 * rb + 8 * g); };
    // residual and row sums, 16 rows at a time (the scheduling barriers here
    // and below keep the compiler from holding more rows' loads and masks than
    // there are registers)
    float sv[16];
    auto res_issue = [&](int p) {
#pragma unroll
        for (int r = 0; r < 8; r++) {
            const int m = min(wrow + 8 * p + r, mlim - 1);
            if (lane < WCOL / 4)
                lds_load16(a.res + (m0 + m) * NT + ncol + 4 * lane,
                           __builtin_amdgcn_readfirstlane(wlds + (p & 1) * WB + r * WP * 4));
        }
    };
    constexpr int CPR = WCOL / 16, RPI = 64 / CPR;  // 16-byte pieces of a row of codes, rows per load
    if (!TOK) {
        res_issue(0);
        res_issue(1);
    } else {
        // all the wave's rows of codes at once, WCOL bytes each
        const int lr = lane / CPR, lc = (lane - lr * CPR) * 16;
#pragma unroll
        for (int r0 = 0; r0 < 32 * RB; r0 += RPI) {
            const int r = r0 + lr;
            if (lr < RPI && r < 32 * RB)
                lds_load16(a.res_codes + (int64_t)tok_id[wrow + r] * NT + ncol + lc,
                           __builtin_amdgcn_readfirstlane(wlds + r0 * WCOL));
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int p = 4 * rb + g;
            if (!TOK) {
                if (p + 1 < 4 * RB) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
                else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                const float* buf = wbuf + (p & 1) * (WB / 4);
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int cb = 0; cb < CB; cb++)
                        acc[rb][cb][4 * g + e] =
                            fadd_rn(acc[rb][cb][4 * g + e], buf[(4 * hf + e) * WP + 32 * cb + l32]);
                if (p + 2 < 4 * RB) {
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the piece is read
                    res_issue(p + 2);
                }
            } else {
                const float4 sc = *(const float4*)(tok_sc + lrow + 32 * rb + 8 * g);
                const float scs[4] = {sc.x, sc.y, sc.z, sc.w};
                const int8_t* x = (const int8_t*)wbuf + (32 * rb + 8 * g + 4 * hf) * WCOL + l32;
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int cb = 0; cb < CB; cb++)
                        acc[rb][cb][4 * g + e] =
                            fadd_rn(acc[rb][cb][4 * g + e], fmul_rn((float)x[e * WCOL + 32 * cb], scs[e]));
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                sv[4 * g + e] = acc[rb][0][4 * g + e];
#pragma unroll
                for (int cb = 1; cb < CB; cb++) sv[4 * g + e] = fadd_rn(sv[4 * g + e], acc[rb][cb][4 * g + e]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        part[cg * MT + row_of(rb, l32 & 15)] = half_sums(sv, l32);
    }
    __syncthreads();
    if (tid < MT) {
        float t = part[tid];
#pragma unroll
        for (int c = 1; c < TL::CG; c++) t = fadd_rn(t, part[c * MT + tid]);
        rowv[tid] = fdiv_rn(t, (float)NT);  // mean
    }
    __syncthreads();
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const float4 mean = row4(rb, g);
            const float mv[4] = {mean.x, mean.y, mean.z, mean.w};
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int cb = 0; cb < CB; cb++) acc[rb][cb][4 * g + e] = fsub_rn(acc[rb][cb][4 * g + e], mv[e]);
            __builtin_amdgcn_sched_barrier(0);
        }
    if (EPI == ENC_EPI_LN) {
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                sv[r] = 0.0f;
#pragma unroll
                for (int cb = 0; cb < CB; cb++) sv[r] = __fmaf_rn(acc[rb][cb][r], acc[rb][cb][r], sv[r]);
            }
            part[cg * MT + row_of(rb, l32 & 15)] = half_sums(sv, l32);
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
        // normalizeRows after a layernorm: the layernorm's factor cancels, a
        // row of deviations over its norm (f64 sum of squares as the
        // reference's norm) is the same row with fewer roundings -- except
        // where the layernorm's f32 variance overflows: its factor is then 0,
        // and so is the row (a deviation that is itself infinite: NaN)
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
            double ds[16];
#pragma unroll
            for (int r = 0; r < 16; r++) {
                ds[r] = 0.0;
#pragma unroll
                for (int cb = 0; cb < CB; cb++) {
                    const double v = (double)acc[rb][cb][r];
                    ds[r] = __fma_rn(v, v, ds[r]);
                }
            }
            dpart[cg * MT + row_of(rb, l32 & 15)] = half_sums(ds, l32);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __syncthreads();
    if (tid < MT) {
        if (EPI == ENC_EPI_LN) {
            float t = part[tid];
#pragma unroll
            for (int c = 1; c < TL::CG; c++) t = fadd_rn(t, part[c * MT + tid]);
            rowv[tid] = (float)(1.0 / sqrt((double)fdiv_rn(t, (float)NT) + 1e-5));
        } else {
            double t = dpart[tid];
#pragma unroll
            for (int c = 1; c < TL::CG; c++) t += dpart[c * MT + tid];
            if (!(t > 0.0)) rowv[tid] = (float)t;  // 0 or NaN
            else if ((float)t < __builtin_inff()) rowv[tid] = fminf((float)(1.0 / sqrt(t)), 3.4e38f);
            else rowv[tid] = t < __builtin_inf() ? 0.0f : __builtin_nanf("");
        }
    }
    __syncthreads();
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const float4 inv = row4(rb, g);
            const float iv[4] = {inv.x, inv.y, inv.z, inv.w};
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int cb = 0; cb < CB; cb++) acc[rb][cb][4 * g + e] = fmul_rn(acc[rb][cb][4 * g + e], iv[e]);
            __builtin_amdgcn_sched_barrier(0);
        }
    if (EPI == ENC_EPI_LN) {
        float* y = a.Y + m0 * NT;
        uint16_t* y16 = a.Y16 + m0 * NT;
        rows_out([&](int m, int c, float4 v) {
            *(float4*)(y + m * NT + c) = v;
            const h4 o = {(_Float16)v.x, (_Float16)v.y, (_Float16)v.z, (_Float16)v.w};
            *(h4*)(y16 + m * NT + c) = o;
        });
        return;
    }
    // masked column sums of each sequence's share of the wave's rows (its
    // slab), one slot after the other from the sequence the slab begins in
    constexpr int WR = 32 * RB;
    const int64_t srow = m0 + WR * rg;  // the slab's first row
    if (srow >= a.M) return;
    const int64_t mr = srow + (lane < WR ? lane : 0);
    const uint64_t live = __ballot(lane < WR && mr < a.M && a.mask[mr < a.M ? mr : 0] != 0);
    const int64_t slab = srow / WR;
    const int64_t seq0 = srow / a.T;
    const int64_t end = srow + WR < a.M ? srow + WR : a.M;
    for (int slot = 0; (seq0 + slot) * a.T < end; slot++) {
        const int64_t f = (seq0 + slot) * a.T - srow;  // the sequence's rows within the slab
        const int lo = f > 0 ? (int)f : 0;
        const int hi = f + a.T < WR ? (int)(f + a.T) : WR;
        const uint64_t upto = hi == 64 ? ~0ull : (1ull << hi) - 1;
        const uint64_t m64 = live & upto & ~((1ull << lo) - 1);
        float sum[CB];
#pragma unroll
        for (int cb = 0; cb < CB; cb++) sum[cb] = 0.0f;
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
            const uint32_t m32 = (uint32_t)(m64 >> (32 * rb + 4 * hf));
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const bool in = (m32 >> (8 * (r >> 2) + (r & 3))) & 1u;
#pragma unroll
                for (int cb = 0; cb < CB; cb++) sum[cb] = in ? fadd_rn(sum[cb], acc[rb][cb][r]) : sum[cb];
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int cb = 0; cb < CB; cb++) {
            const float t = fadd_rn(sum[cb], __shfl_xor(sum[cb], 32));
            if (hf == 0) a.Y[(slab * a.slots + slot) * NT + nb + 32 * cb] = t;
        }
    }
}

template <int MT, int NT, int EPI, bool TOK>
static hipError_t launch_enc_gemm16_one(const EncGemmArgs& a, hipStream_t s) {
    const int64_t rt = (a.M + MT - 1) / MT, ctn = a.N / NT;
    const int64_t grid = (rt + 7) / 8 * 8 * ctn;
    if (grid > 0x7FFFFFFF) return hipErrorInvalidValue;
    const size_t lds = EncTile<MT, NT>::LDS;
    static bool attr = false;
    if (!attr) {
        hipError_t e = hipFuncSetAttribute((const void*)enc_gemm16_kernel<MT, NT, EPI, TOK>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        attr = true;
    }
    hipLaunchKernelGGL((enc_gemm16_kernel<MT, NT, EPI, TOK>), dim3((unsigned)grid), dim3(512), lds, s, a);
    return hipGetLastError();
}

template <int MT, int NT, int EPI>
static hipError_t launch_enc_gemm16_tok(const EncGemmArgs& a, hipStream_t s) {
    if constexpr (EPI == ENC_EPI_LN) {
        if (!a.res) return launch_enc_gemm16_one<MT, NT, EPI, true>(a, s);
    }
    return launch_enc_gemm16_one<MT, NT, EPI, false>(a, s);
}

template <int MT, int EPI>
static hipError_t launch_enc_gemm16_nt(int nt, const EncGemmArgs& a, hipStream_t s) {
    if (nt == 384) return launch_enc_gemm16_tok<MT, 384, EPI>(a, s);
    if (nt == 256) return launch_enc_gemm16_tok<MT, 256, EPI>(a, s);
    return launch_enc_gemm16_tok<MT, 128, EPI>(a, s);
}

// The 256-row tile once it gives every second CU a workgroup; fewer rows take
// 64-row tiles.
static bool enc_gemm16_big(int64_t M, int N, int nt) { return (M + 255) / 256 * (N / nt) >= 128; }

template <int EPI>
static hipError_t launch_enc_gemm16_epi(int nt, const EncGemmArgs& a, hipStream_t s) {
    return enc_gemm16_big(a.M, a.N, nt) ? launch_enc_gemm16_nt<256, EPI>(nt, a, s)
                                        : launch_enc_gemm16_nt<64, EPI>(nt, a, s);
}

int enc_pool_slab(int64_t M, int64_t d) { return enc_gemm16_big(M, (int)d, (int)d) ? 64 : 32; }

bool enc_ln_fused(int64_t d) { return d == 128 || d == 256 || d == 384; }

hipError_t launch_enc_gemm16(int epi, const EncGemmArgs& a, hipStream_t s) {
    const int w = epi == ENC_EPI_F32 ? a.D : a.N;  // the column tile divides an output matrix's width
    if (a.M <= 0 || a.K <= 0 || a.K % 32 != 0 || w <= 0 || w % 128 != 0 || a.N % w != 0) return hipErrorInvalidValue;
    const int nt = w % 384 == 0 ? 384 : (w % 256 == 0 ? 256 : 128);
    if ((epi == ENC_EPI_LN || epi == ENC_EPI_LN_POOL) && nt != a.N) return hipErrorInvalidValue;
    if (epi == ENC_EPI_LN_POOL && !a.res) return hipErrorInvalidValue;
    switch (epi) {
        case ENC_EPI_F32: return launch_enc_gemm16_epi<ENC_EPI_F32>(nt, a, s);
        case ENC_EPI_GELU16: return launch_enc_gemm16_epi<ENC_EPI_GELU16>(nt, a, s);
        case ENC_EPI_LN: return launch_enc_gemm16_epi<ENC_EPI_LN>(nt, a, s);
        default: return launch_enc_gemm16_epi<ENC_EPI_LN_POOL>(nt, a, s);
    }
}

// ------------------------------------------------------------------ attention

// softmax(q k^T) v for up to 64 query rows of one sequence of T <= 64*NK
// positions, f32 on the matrix cores (v_mfma_f32_32x32x2f32), f16 out: grid
// (ceil(T / 64), sequences), 8 waves.  D = 128*CW.
//   1. S = q k^T, one or two 32 x 32 tiles a wave: 32 columns of the q and k
//      rows at a time through a ring of three LDS stages (direct-to-LDS loads,
//      a row's 16-byte column c stored at c ^ (row & 7)); a 16-byte piece of a
//      row is four steps of an operand (half wave h takes columns 8i + 4h + e
//      at step e, on both sides).
//   2. softmax of the rows of S in LDS, 16 lanes a row: f64 exponentials and
//      sum, as softmaxRows.
//   3. P v: 32*CW columns for one row block a wave, P from LDS in the same
//      order of t, v rows straight from memory (one 128-byte piece per half
//      wave, two steps ahead).
// The separate score product, softmax and value product moved the scores, an
// f32 copy of the result and every operand through HBM: 165 us against
// 107 for 1024 sequences of 64, d = 384 (the three reads alone are 61 us at
// the copy rate; with the q and k rows read straight into registers, 16 bytes
// a lane and row, 140).
template <int CW, int NK>
struct AttTile {
    static constexpr int STAGE = (64 + 64 * NK) * 128, NST = 3;
    static constexpr int L = 1 + NK;  // 1 KB loads (8 rows) per wave and stage
    static constexpr int LD = 64 * NK + 4;
    static constexpr size_t LDS = (size_t)NST * STAGE > (size_t)64 * LD * 4 ? (size_t)NST * STAGE : (size_t)64 * LD * 4;
};

template <int CW, int NK>
__global__ __launch_bounds__(512, NK == 1 ? 4 : 2) void enc_attention_kernel(const float* __restrict__ q,
                                                                             const float* __restrict__ k,
                                                                             const float* __restrict__ v, int T,
                                                                             uint16_t* __restrict__ out) {
    typedef AttTile<CW, NK> TL;
    constexpr int D = 128 * CW, L = TL::L, NST = TL::NST, LD = TL::LD, Tp = 64 * NK;
    extern __shared__ __attribute__((aligned(16))) float S[];  // the stages, then [64][LD]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l32 = lane & 31, hf = lane >> 5;
    const int64_t row0 = (int64_t)blockIdx.y * T;  // the sequence's first row
    const int q0 = blockIdx.x * 64;
    const int rb = wave & 1;
    const bool mine = q0 + 32 * rb < T;  // the wave's row block holds rows

    {
        const uint8_t* src[L];
        const int lr = lane >> 3;
#pragma unroll
        for (int u = 0; u < L; u++) {
            const int sg = wave * L + u;  // segments 0..7: q rows, then k rows
            const int r = sg < 8 ? q0 + 8 * sg + lr : 8 * (sg - 8) + lr;
            src[u] = (const uint8_t*)((sg < 8 ? q : k) + (row0 + (r < T ? r : T - 1)) * D) + ((lane & 7) ^ lr) * 16;
        }
        const uint32_t base =
            __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)S);
        auto issue = [&](int kc, int st) {
            const uint32_t d = __builtin_amdgcn_readfirstlane(base + st * TL::STAGE + wave * L * 1024);
#pragma unroll
            for (int u = 0; u < L; u++) lds_load16(src[u] + kc * 128, d + u * 1024);
        };
        constexpr int nk = D / 32, NC = (2 * NK + 3) / 4;
        issue(0, 0);
        issue(1, 1);
        const int cq = wave >> 1;  // column blocks cq and cq + 4
        f16v acc[NC];
#pragma unroll
        for (int j = 0; j < NC; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[j][r] = 0.0f;
        int st = 0;
        for (int kc = 0; kc < nk; kc++, st = st == NST - 1 ? 0 : st + 1) {
            wait_barrier<L, NST - 2>(nk - 1 - kc);
            if (kc + NST - 1 < nk) issue(kc + NST - 1, st == 0 ? NST - 1 : st - 1);
            const uint8_t* Q = (const uint8_t*)S + st * TL::STAGE + (32 * rb + l32) * 128;
            const uint8_t* Kt = (const uint8_t*)S + st * TL::STAGE + (64 + l32) * 128;
            if (!mine) continue;
#pragma unroll
            for (int j = 0; j < NC; j++) {
                const int cb = cq + 4 * j;
                if (cb >= 2 * NK || 32 * cb >= T) continue;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int c = ((2 * i + hf) ^ (l32 & 7)) * 16;
                    const float4 av = *(const float4*)(Q + c), bv = *(const float4*)(Kt + 32 * cb * 128 + c);
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av.x, bv.x, acc[j], 0, 0, 0);
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av.y, bv.y, acc[j], 0, 0, 0);
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av.z, bv.z, acc[j], 0, 0, 0);
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av.w, bv.w, acc[j], 0, 0, 0);
                }
            }
        }
        __syncthreads();  // every wave is done with the stages
#pragma unroll
        for (int j = 0; j < NC; j++) {
            const int cb = cq + 4 * j;
            if (cb >= 2 * NK) continue;
#pragma unroll
            for (int r = 0; r < 16; r++)
                S[(32 * rb + 8 * (r >> 2) + 4 * hf + (r & 3)) * LD + 32 * cb + l32] = acc[j][r];
        }
    }
    __syncthreads();
    // 16 lanes a row, four rows a wave at a time, the wave's next four after
    // them; lane i takes columns 4i + 64j .. + 3
    const int i16 = lane & 15;
#pragma unroll
    for (int it = 0; it < 2; it++) {
        const int r = 32 * it + 4 * wave + (lane >> 4);
        if (q0 + 32 * it >= T) break;  // (rows past T in a block that holds some: values nobody stores)
        float* s = S + r * LD + 4 * i16;
        float4 x[4];
        float m = -__builtin_inff();
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (64 * j >= Tp) break;
            const int c = 4 * i16 + 64 * j;
            x[j] = float4{-__builtin_inff(), -__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
            if (c < Tp) x[j] = *(const float4*)(s + 64 * j);
            if (c >= T) x[j].x = -__builtin_inff();
            if (c + 1 >= T) x[j].y = -__builtin_inff();
            if (c + 2 >= T) x[j].z = -__builtin_inff();
            if (c + 3 >= T) x[j].w = -__builtin_inff();
            m = fmaxf(m, fmaxf(fmaxf(x[j].x, x[j].y), fmaxf(x[j].z, x[j].w)));
        }
        m = row16_max(m);
        double sum = 0.0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (64 * j >= Tp) break;
            const int c = 4 * i16 + 64 * j;
            const double e0 = c < T ? exp((double)fsub_rn(x[j].x, m)) : 0.0;
            const double e1 = c + 1 < T ? exp((double)fsub_rn(x[j].y, m)) : 0.0;
            const double e2 = c + 2 < T ? exp((double)fsub_rn(x[j].z, m)) : 0.0;
            const double e3 = c + 3 < T ? exp((double)fsub_rn(x[j].w, m)) : 0.0;
            x[j] = float4{(float)e0, (float)e1, (float)e2, (float)e3};
            sum += (e0 + e1) + (e2 + e3);
        }
        sum = row16_sum(sum);
        const float inv = sum == 0.0 ? 1.0f : (float)(1.0 / sum);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (64 * j >= Tp) break;
            if (4 * i16 + 64 * j < Tp)
                *(float4*)(s + 64 * j) = float4{fmul_rn(x[j].x, inv), fmul_rn(x[j].y, inv), fmul_rn(x[j].z, inv),
                                                fmul_rn(x[j].w, inv)};
        }
    }
    __syncthreads();
    if (!mine) return;
    f16v acc[CW];
#pragma unroll
    for (int w = 0; w < CW; w++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[w][r] = 0.0f;
    const int c0 = (wave >> 1) * 32 * CW + l32;
    const float* vb = v + row0 * D + c0;
    auto load = [&](float (&dst)[4][CW], int i) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int t = 8 * i + 4 * hf + e;
#pragma unroll
            for (int w = 0; w < CW; w++) dst[e][w] = t < T ? vb[t * D + 32 * w] : 0.0f;
        }
    };
    // two steps of v in flight ahead of the one multiplied
    float bv[3][4][CW];
    const int steps = (T + 7) / 8;
    load(bv[0], 0);
    load(bv[1], 1);
    for (int i0 = 0; i0 < steps; i0 += 3) {
#pragma unroll
        for (int u = 0; u < 3; u++) {
            const int i = i0 + u;
            if (i >= steps) break;
            load(bv[(u + 2) % 3], i + 2);
            const float4 p = *(const float4*)(S + (32 * rb + l32) * LD + 8 * i + 4 * hf);
            const float pa[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int w = 0; w < CW; w++)
                    acc[w] = __builtin_amdgcn_mfma_f32_32x32x2f32(pa[e], bv[u][e][w], acc[w], 0, 0, 0);
        }
    }
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int t = q0 + 32 * rb + 8 * (r >> 2) + 4 * hf + (r & 3);
        if (t >= T) continue;
#pragma unroll
        for (int w = 0; w < CW; w++) out[(row0 + t) * D + c0 + 32 * w] = f2h(acc[w][r]);
    }
}

bool enc_attention_supported(int64_t t, int64_t d) { return t >= 1 && t <= 256 && d % 128 == 0 && d >= 128 && d <= 512; }

template <int CW, int NK>
static hipError_t launch_enc_attention_one(const float* q, const float* k, const float* v, int64_t b, int t,
                                           uint16_t* out, hipStream_t s) {
    const size_t lds = AttTile<CW, NK>::LDS;
    static bool attr = false;
    if (!attr) {
        hipError_t e = hipFuncSetAttribute((const void*)enc_attention_kernel<CW, NK>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        attr = true;
    }
    hipLaunchKernelGGL((enc_attention_kernel<CW, NK>), dim3((unsigned)((t + 63) / 64), (unsigned)b), dim3(512), lds, s,
                       q, k, v, t, out);
    return hipGetLastError();
}

template <int CW>
static hipError_t launch_enc_attention_cw(const float* q, const float* k, const float* v, int64_t b, int t,
                                          uint16_t* out, hipStream_t s) {
    switch ((t + 63) / 64) {
        case 1: return launch_enc_attention_one<CW, 1>(q, k, v, b, t, out, s);
        case 2: return launch_enc_attention_one<CW, 2>(q, k, v, b, t, out, s);
        case 3: return launch_enc_attention_one<CW, 3>(q, k, v, b, t, out, s);
        default: return launch_enc_attention_one<CW, 4>(q, k, v, b, t, out, s);
    }
}

hipError_t launch_enc_attention(const float* q, const float* k, const float* v, int64_t b, int t, int d,
                                uint16_t* out, hipStream_t s) {
    if (!enc_attention_supported(t, d) || b <= 0 || b > 65535) return hipErrorInvalidValue;
    switch (d / 128) {
        case 1: return launch_enc_attention_cw<1>(q, k, v, b, t, out, s);
        case 2: return launch_enc_attention_cw<2>(q, k, v, b, t, out, s);
        case 3: return launch_enc_attention_cw<3>(q, k, v, b, t, out, s);
        default: return launch_enc_attention_cw<4>(q, k, v, b, t, out, s);
    }
}

// ----------------------------------------------------------------------- pool

namespace {

// Unmasked positions of a sequence, counted by the whole workgroup.
__device__ __forceinline__ int masked_count(const int32_t* mk, int T, int* cnt) {
    int n = 0;
    for (int t = threadIdx.x; t < T; t += 256) n += mk[t] != 0 ? 1 : 0;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) n += __shfl_xor(n, off);
    if ((threadIdx.x & 63) == 0) cnt[threadIdx.x >> 6] = n;
    __syncthreads();
    return cnt[0] + cnt[1] + cnt[2] + cnt[3];
}

}  // namespace

// Mean of a sequence from the slabs' column sums (ENC_EPI_LN_POOL), in row
// order, and the f16 output; one workgroup per sequence.
__global__ __launch_bounds__(256) void enc_pool_slabs_kernel(const float* __restrict__ P,
                                                             const int32_t* __restrict__ mask, int T, int d, int slab,
                                                             int slots, uint16_t* __restrict__ out) {
    __shared__ int cnt[4];
    const int64_t b = blockIdx.x;
    const int count = masked_count(mask + b * T, T, cnt);
    const float inv = count ? 1.0f / (float)count : 0.0f;
    const int64_t s0 = b * T / slab, s1 = (b * T + T - 1) / slab;
    for (int c = threadIdx.x; c < d; c += 256) {
        float v = 0.0f;
        for (int64_t s = s0; s <= s1; s++) v = v + P[(s * slots + (b - s * slab / T)) * d + c];
        out[b * d + c] = f2h(count ? v * inv : 0.0f);
    }
}

hipError_t launch_enc_pool_slabs(const float* P, const int32_t* mask, int64_t b, int t, int d, int slab, int slots,
                                 uint16_t* out, hipStream_t s) {
    hipLaunchKernelGGL(enc_pool_slabs_kernel, dim3((unsigned)b), dim3(256), 0, s, P, mask, t, d, slab, slots, out);
    return hipGetLastError();
}

}  // namespace manta
