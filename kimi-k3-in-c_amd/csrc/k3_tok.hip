/* SPDX-License-Identifier: Apache-2.0 */
/*
 * k3_tok.hip -- dense products of several tokens, fp32-accurate, on the matrix cores:
 * Y[t][r] = sum_k W[r][k] * x[t][k] for two tokens and more, bf16 or fp32 weights, fp32
 * activations straight from the caller (k3_matmul_bf16 / k3_matmul of the reference,
 * src/core/k3_ops.c:1108-1213, 265-291, applied to each token).
 *
 * A vector-unit GEMV that reads the weights once per four tokens and spends a vector FMA per
 * product took, for 7168 -> 3584 in bf16, 13 / 22 / 94 / 153 / 607 us at 4 / 8 / 37 / 64 / 256
 * tokens (fp32: 18 / 33 / - / 222 / 876). Here a weight is read once per block of up to 64
 * tokens and the products run on the matrix cores: 10.5 / 11.2 / 20.8 / 25 / 55 us (fp32: 17.2
 * / 17.6 / - / 38 / 144).
 *
 *   bf16 weights: x is cut into three bf16 terms by truncation, x = h + m + l. Each cut
 *     keeps the next 8 significand bits, so the three terms hold all 24 and every product
 *     with a weight is exact; v_mfma_f32_16x16x32_bf16 adds the three into one fp32 sum.
 *     (Two rounded terms, as the expert kernels use, would lose 7 bits.) bf16 ends at 2^-133,
 *     so bits of x below that are dropped: only an |x| under 2^-109 has any.
 *   fp32 weights: v_mfma_f32_16x16x4_f32 on the values as they are.
 *   MXFP4 weights (k3_matmul_mxfp4 of the reference for three tokens and more): the codes are
 *     exact in bf16 under their block's scale; x comes as two rounded bf16 terms, or one where
 *     the entry point's caller asked for that (the other's products are of zeros: a kernel
 *     without them would save little, the weights and x bound it). The expert streaming kernel, which reads the weights once per 16 or 32
 *     tokens through a register ring, took 16 / 39 / 273 us for 7168 -> 2048 at 8 / 64 / 512
 *     tokens and 3575 at 512 of 12288 -> 16384; here 11.5 / 22 / 54 and 635. K of any multiple
 *     of 32: the scales come a byte at a time, since a row's start is at no multiple of 4 (dwords
 *     where K % 128 == 0: 11.1 / 21 / 52 and 617, not worth a second kernel).
 *
 * A workgroup owns MT tiles of 16 rows x N8 groups of 8 tokens; its KW waves split K, and no
 * barrier joins them until their sums meet in LDS (added in wave order, so the result does
 * not depend on timing). A wave walks its share 32 columns a stage: the buffer unit copies the
 * stage's weights and fp32 activations into LDS of the wave's own (ST stages, all but one in
 * flight), consecutive lanes reading consecutive bytes of a row, and the wave reads its
 * fragments back from there. Loading the fragments straight into registers instead, where
 * neighbouring lanes belong to different rows and the L1 works a line per lane, took 41 us at
 * 64 tokens of 7168 -> 3584 and 78 at 256; the stages through registers into LDS, 24 and 67.
 * A 16-byte piece p of row r lies at piece p ^ (r / RL mod PR) of its row (RL rows to 256
 * bytes, PR pieces to a row), so the 16 rows of a fragment read cover the 64 banks once. The
 * contraction order inside a stage is free as long as both operands agree: lane group g takes
 * columns 8g .. 8g+7. No scratch memory: the entry points have none to give, so K cannot be
 * split over workgroups, and every row block reads all of its tokens' x.
 *
 * What bounds it: for few tokens the weight stream, the fill of the stages and the adding up; from
 * about 16 tokens no unit by itself (counters: 14-29 bytes a cycle and CU through the L1, whose width is
 * 64; matrix pipes busy 26-28 % of the cycles in large bf16 and MXFP4 products, vector issue 34-40 %;
 * 55 and 24 % for fp32 weights, whose matrix rate is 1/16), but the chain of a wave's stage -- its
 * copies' arrival, the LDS reads, the cut (5.5 vector instructions per element; with v_dot2_f32_bf16,
 * 3.5, nothing changed) or dequantisation, the products -- since the LDS holds one or two waves to a
 * SIMD. The launch rule (tok_cost) weighs these.
 *
 * Infinities and NaN: the cut of an infinite x, or a zero term against an infinite weight,
 * gives NaN where the product of the uncut values is infinite. Finite operands give none, so
 * a NaN in the sum is the sign of such a case, and that element is recomputed with plain
 * FMAs, by the whole wave -- unless its token, or its weight row, holds a NaN: each such row is
 * looked through once. 64 tokens of 7168 -> 3584 in bf16, 27 us: one token all NaN (padding) 30, a
 * NaN at the end of one 49, in a weight row 103, an infinity in a token (3584 dot products)
 * 1.6 ms; by single lanes, one dot product after another, 5.3 ms for each.
 */
#include "k3_common.h"
#include "k3k.h"

#include <type_traits>
#include <utility>

namespace {

template <typename F, int... S>
__device__ __forceinline__ void k3_tok_for_impl(F &&f, std::integer_sequence<int, S...>)
{
    (f(std::integral_constant<int, S>{}), ...);
}
/* f(std::integral_constant<int, s>{}) for s = 0 .. N-1, unrolled */
template <int N, typename F>
__device__ __forceinline__ void k3_tok_for(F &&f)
{
    k3_tok_for_impl(f, std::make_integer_sequence<int, N>{});
}

typedef uint32_t k3_u32x4 __attribute__((ext_vector_type(4)));

enum { TOK_F32 = 0, TOK_BF16 = 1, TOK_MX = 2 };       /* weights */

struct TokArgs {
    float *y;
    const float *x;                       /* fp32 activations, or */
    const uint16_t *xhi;                  /* their two bf16 terms, lo_off bytes apart */
    uint32_t lo_off;                      /* (0: one term, the other reads as zeros) */
    const void *W, *W2;                   /* W2: GLU's up matrix */
    const uint8_t *scales;                /* MX */
    int in, out, ntok, ldy, accumulate;
    int act, rpt;                         /* GLU: activation, rows of each matrix per workgroup */
    float b1, b2;
    int ntt, items, per_xcd;              /* token blocks, workgroups with work, per XCD */
};

/* The NaN case, by a whole wave. Whether a row of n values holds a NaN: */
template <int BF>
__device__ __forceinline__ bool tok_row_nan(const void *row, int n)
{
    const int lane = threadIdx.x & 63;
    for (int k0 = 0; k0 < n; k0 += 64 * 8) {
        bool nan = false;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int k = k0 + 64 * i + lane;
            const float f = k >= n ? 0.0f : BF ? k3_bf16_to_f32(((const uint16_t *)row)[k]) : ((const float *)row)[k];
            nan |= f != f;
        }
        if (__ballot(nan)) return true;
    }
    return false;
}

/* and the plain product of one output (every lane has it) */
template <int BF>
__device__ __forceinline__ float tok_plain_dot(const void *W, const float *x, int in)
{
    const int lane = threadIdx.x & 63;
    float s = 0.0f;
    for (int k0 = 0; k0 < in; k0 += 64 * 8) {
        float wq[8], xq[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int k = min(k0 + 64 * i + lane, in - 1);
            wq[i] = BF ? k3_bf16_to_f32(((const uint16_t *)W)[k]) : ((const float *)W)[k];
            xq[i] = x[k];
        }
#pragma unroll
        for (int i = 0; i < 8; i++) s = k0 + 64 * i + lane < in ? fmaf(wq[i], xq[i], s) : s;
    }
    for (int m = 32; m > 0; m >>= 1) s += __shfl_xor(s, m, 64);
    return s;
}

/* The NaN sums of a workgroup (mt x nb tiles, a 4 x 1 piece per lane) in s, recomputed where no
 * operand row holds a NaN; W2 (GLU): the second tile's weights. tok: the workgroup's tokens. */
template <int BF>
__device__ __noinline__ void tok_recompute(k3_f32x4 *s, const char *W, const char *W2, size_t wrow, const float *x, int in,
                                           int nrow, int ntok, int mt, int nb)
{
    const int lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
    uint64_t xseen = 0, xnan = 0;                  /* tokens looked at, those with a NaN */
    for (int m = 0; m < mt; m++) {
        const char *w = W2 && m ? W2 : W;
        const int r0 = W2 ? 0 : 16 * m;
        uint32_t wseen = 0, wnan = 0;              /* rows of the tile */
        for (int b = 0; b < nb; b++) {
            k3_f32x4 v = s[(m * nb + b) * 64 + lane];
            uint32_t need = 0;
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (v[e] != v[e] && 16 * b + r16 < ntok && r0 + 4 * g + e < nrow) need |= 1u << e;
            while (const uint64_t left = __ballot(need != 0)) {
                /* one element of the first lane that has any: token t, row r of the tile */
                const int from = __ffsll((unsigned long long)left) - 1;
                const int e1 = __ffs(__builtin_amdgcn_readlane((int)need, from)) - 1;
                const int t = 16 * b + (from & 15), r = 4 * (from >> 4) + e1;
                const float *xr = x + (size_t)t * in;
                const char *wr = w + (size_t)(r0 + r) * wrow;
                if (!((xseen >> t) & 1)) {
                    xseen |= 1ull << t;
                    if (tok_row_nan<0>(xr, in)) xnan |= 1ull << t;
                }
                if ((xnan >> t) & 1) {
                    if (r16 == (from & 15)) need = 0;
                    continue;
                }
                if ((wnan >> r) & 1) {
                    if (g == from >> 4) need &= ~(1u << e1);
                    continue;
                }
                const float p = tok_plain_dot<BF>(wr, xr, in);
                if (p != p && !((wseen >> r) & 1)) {
                    wseen |= 1u << r;
                    if (tok_row_nan<BF>(wr, in)) wnan |= 1u << r;
                }
                if (lane == from) {
                    need &= ~(1u << e1);
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = e == e1 ? p : v[e];
                }
            }
            s[(m * nb + b) * 64 + lane] = v;
        }
    }
}

/* eight floats -> their three bf16 terms by truncation */
__device__ __forceinline__ void tok_cut(k3_u32x4 a, k3_u32x4 b, uint4 &h, uint4 &m, uint4 &l)
{
    const uint32_t u[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint32_t r[8], q[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const float t = __uint_as_float(u[e]) - __uint_as_float(u[e] & 0xFFFF0000u);
        r[e] = __float_as_uint(t);
        q[e] = __float_as_uint(t - __uint_as_float(r[e] & 0xFFFF0000u));
    }
    /* the upper halves of two words in one */
    auto up = [](uint32_t lo, uint32_t hi) { return __builtin_amdgcn_perm(hi, lo, 0x07060302u); };
    h = make_uint4(up(u[0], u[1]), up(u[2], u[3]), up(u[4], u[5]), up(u[6], u[7]));
    m = make_uint4(up(r[0], r[1]), up(r[2], r[3]), up(r[4], r[5]), up(r[6], r[7]));
    l = make_uint4(up(q[0], q[1]), up(q[2], q[3]), up(q[4], q[5]), up(q[6], q[7]));
}

/* eight floats -> one bf16 term each, to nearest even (v_cvt_pk_bf16_f32; 8 tokens of 7168 -> 2048
 * through the shared expert 20.2 us, 24.0 with k3_bf16_rne, three terms 21.7) */
__device__ __forceinline__ uint4 tok_round(k3_u32x4 a, k3_u32x4 b)
{
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef __bf16 h2 __attribute__((ext_vector_type(2)));
    const uint32_t u[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint32_t p[4];
#pragma unroll
    for (int e = 0; e < 4; e++)
        p[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{__uint_as_float(u[2 * e]), __uint_as_float(u[2 * e + 1])}), h2));
    return make_uint4(p[0], p[1], p[2], p[3]);
}

/* Stages of 32 columns. WT: the weights' type; XT 0: fp32 activations, 1: two bf16 terms, 2: fp32, and
 * any K and alignment: a piece may start at any element, so it is loaded into registers (a stage
 * ahead) and stored into LDS, and the stage that K ends in is loaded by elements; 64 tokens of
 * 7169 -> 3584 47 us in bf16, 4044 on a wave per row and token, 25 aligned.
 * GLU: tiles 0 and 1 are rpt rows of W and the same rows of W2, y = act(tile 0, tile 1). GLU 2: x
 * is rounded to one bf16 term, and so is y (stored as fp32, whose cut is that term and zeros): the
 * one-term precision of the shared expert.
 * WT MX: the codes come 128 columns at a time (a piece is a block of 32) into buffers of their
 * own, one chunk ahead, and their scale bytes into registers (lane: row r16, block g; a permute
 * hands a stage's to its rows' lanes); lane group g takes dword g of the block a stage
 * multiplies, which is columns 8g .. 8g+7. */
template <int WT, int XT, int GLU, int MT, int N8, int KW, int ST>
__global__ __launch_bounds__(64 * KW) void tok_gemm_kernel(TokArgs a)
{
    constexpr int NB = (N8 + 1) / 2;               /* matrix column blocks of 16 tokens */
    constexpr int BF = WT != TOK_F32, MX = WT == TOK_MX;
    constexpr int ES = WT == TOK_F32 ? 4 : 2;      /* bytes per weight (not MX) */
    constexpr int PRW = 2 * ES, PRX = 8;           /* 16-byte pieces per row and stage */
    constexpr int RLW = 16 / PRW, RLX = 2;         /* rows to 256 bytes of LDS */
    constexpr int SLW = MX ? 0 : 16 * PRW;         /* slots per row tile (64 per token group) */
    constexpr int WSL = MT * SLW + N8 * 64;        /* slots per wave and stage */
    constexpr int ND = WSL / 64;                   /* copy instructions per wave and stage */
    constexpr uint32_t OOB = 0x80000000u;
    static_assert(ST >= 2 && ST <= 4 && ND * (ST - 1) < 64, "stages, vmcnt field");
    static_assert(!MX || ST != 3, "eight stages to a loop");
    static_assert(!GLU || (MT == 2 && !MX), "gate and up tiles");
    constexpr int RED = (KW - 1) * MT * NB * 64;   /* the waves' sums, in stage array 0 */
    constexpr int B0 = RED > KW * WSL ? RED : KW * WSL;
    /* an array per stage of a plain vector type, read at one integer index: the compiler then
     * tells a copy into one array from reads of another (through longer pointer chains it does
     * not, and waits for every copy in flight before each read) */
    __shared__ __attribute__((aligned(1024))) k3_u32x4 b0[B0], b1[KW * WSL];
    __shared__ __attribute__((aligned(1024))) k3_u32x4 b2[ST > 2 ? KW * WSL : 1], b3[ST > 3 ? KW * WSL : 1];
    __shared__ __attribute__((aligned(1024))) uint32_t w0[MX ? KW * MT * 256 : 1], w1[MX ? KW * MT * 256 : 1];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int item = (blockIdx.x % K3_NXCD) * a.per_xcd + (int)blockIdx.x / K3_NXCD;
    if (item >= a.items) return;
    const int tb = item % a.ntt, rb = item / a.ntt;
    const int row0 = rb * (GLU ? a.rpt : 16 * MT), tok0 = tb * 8 * N8;
    const int nrow = min(a.out - row0, GLU ? a.rpt : 16 * MT), ntok = min(a.ntok - tok0, 8 * N8);
    const size_t wrow = MX ? (size_t)a.in / 2 : (size_t)a.in * ES;       /* bytes per weight row */
    const k3_rsrc rw = k3_make_rsrc((const char *)a.W + row0 * wrow, (uint32_t)(nrow * wrow));
    const k3_rsrc rw2 = k3_make_rsrc(GLU ? (const char *)a.W2 + row0 * wrow : (const char *)a.W, GLU ? (uint32_t)(nrow * wrow) : 0u);
    const k3_rsrc rs = k3_make_rsrc(MX ? a.scales + (size_t)row0 * (a.in / 32) : nullptr, MX ? (uint32_t)nrow * (uint32_t)(a.in / 32) : 0u);
    const k3_rsrc rx = XT == 1 ? k3_make_rsrc(a.xhi + (size_t)tok0 * a.in, a.lo_off + (uint32_t)ntok * (uint32_t)a.in * 2u)
                          : k3_make_rsrc(a.x + (size_t)tok0 * a.in, (uint32_t)ntok * (uint32_t)a.in * 4u);
    /* the wave's share, whole chunks of MX codes */
    constexpr int U = MX ? 4 : 1;
    const int nst = (a.in + 31) / 32;
    const int nch = (nst + U - 1) / U;
    const int s0 = wv * nch / KW * U, s1 = min((wv + 1) * nch / KW * U, nst);
    /* copy instruction i fills slots 64 i + lane: its lane's source row and piece. Rows and
     * tokens past the end, pieces past K and stages past the share read at 2^31 and more,
     * beyond the buffer: zeros, no data moved. */
    uint32_t voff[ND], col[ND];
#pragma unroll
    for (int i = 0; i < ND; i++) {
        const bool isw = i < MT * SLW / 64;
        const int sl = 64 * i + lane - (isw ? 0 : MT * SLW);
        const int pr = isw ? PRW : PRX, row = sl / pr;
        const int p = (sl % pr) ^ ((row / (isw ? RLW : RLX)) & (pr - 1));
        const int wr = GLU ? row & 15 : row;
        const uint32_t NONE = XT == 2 ? 16u * p : OOB;     /* XT 2: the first row again, for nothing */
        if (isw) {
            voff[i] = wr < nrow ? (uint32_t)wr * (uint32_t)a.in * ES + 16u * p : NONE;
            col[i] = p * (16 / ES);
        } else if (XT == 1) {                      /* pieces 0-3: hi, 4-7: lo */
            voff[i] = row < ntok && (p < 4 || a.lo_off) ? (uint32_t)row * (uint32_t)a.in * 2u + 16u * (p & 3) + (p >> 2) * a.lo_off : OOB;
            col[i] = (p & 3) * 8;
        } else {
            voff[i] = row < ntok ? (uint32_t)row * (uint32_t)a.in * 4u + 16u * p : NONE;
            col[i] = p * 4;
        }
    }
    /* MX: a tile's chunk copy (slot lane: row lane / 4, block mb = (lane % 4) ^ (row / 4 % 4)) */
    const int mb = (lane & 3) ^ ((lane >> 4) & 3);
    const uint32_t mo = (uint32_t)(lane >> 2) * (uint32_t)(a.in / 2) + 16u * mb;
    const uint32_t so = (uint32_t)r16 * (uint32_t)(a.in / 32) + g;
    uint32_t sc[2][MT];
    auto copy_w = [&](int c, auto slot) {
        constexpr int S = decltype(slot)::value;
        const bool inw = 4 * c + mb < s1, ins = 4 * c + g < s1;
#pragma unroll
        for (int m = 0; m < MT; m++) {
            const uint32_t ro = 16u * m;
            uint32_t *d = S ? w1 : w0;
            k3_dma16(rw, &d[(wv * MT + m) * 256], inw && ro + (lane >> 2) < (uint32_t)nrow ? mo + ro * (uint32_t)(a.in / 2) + 64u * c : OOB, 0);
            sc[S][m] = k3_bload1(rs, ins && ro + r16 < (uint32_t)nrow ? so + ro * (uint32_t)(a.in / 32) + 4u * c : OOB);
        }
    };
    auto buf = [&](auto slot) -> k3_u32x4 * {
        constexpr int S = decltype(slot)::value;
        if constexpr (S == 0) return b0;
        else if constexpr (S == 1) return b1;
        else if constexpr (S == 2) return b2;
        else return b3;
    };
    auto copy = [&](int s, auto slot) {
        k3_u32x4 *d = buf(slot);
        const uint32_t left = s < s1 ? (uint32_t)(a.in - 32 * s) : 0u;      /* columns from here */
        const uint32_t ss = (uint32_t)min(s, nst - 1);
#pragma unroll
        for (int i = 0; i < ND; i++) {
            const bool isw = i < MT * SLW / 64, up = GLU && i >= SLW / 64;
            k3_dma16(isw ? (up ? rw2 : rw) : rx, &d[wv * WSL + 64 * i], col[i] < left ? voff[i] : OOB,
                     ss * (32u * (isw ? ES : XT ? 2 : 4)));
        }
    };
    k3_u32x4 reg[XT == 2 ? ND : 1];
    auto fetch = [&](int s) {
        typedef k3_u32x4 any_u32x4 __attribute__((aligned(2)));
        const int left = s < s1 ? a.in - 32 * s : 0;
#pragma unroll
        for (int i = 0; i < ND; i++) {
            const bool isw = i < MT * SLW / 64;
            const char *q = (isw ? (const char *)a.W + row0 * wrow : (const char *)(a.x + (size_t)tok0 * a.in)) + voff[i];
            if (left >= 32) {
                reg[i] = *reinterpret_cast<const any_u32x4 *>(q + (size_t)s * (32 * (isw ? ES : 4)));
            } else {
                q += (size_t)s * (32 * (isw ? ES : 4));
                uint32_t v[4] = {0u, 0u, 0u, 0u};
                if (isw && ES == 2) {
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        if ((int)col[i] + e < left) v[e >> 1] |= (uint32_t)reinterpret_cast<const uint16_t *>(q)[e] << (16 * (e & 1));
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if ((int)col[i] + e < left) v[e] = reinterpret_cast<const uint32_t *>(q)[e];
                }
                reg[i] = k3_u32x4{v[0], v[1], v[2], v[3]};
            }
        }
    };
    auto stash = [&](auto slot) {
        k3_u32x4 *d = buf(slot);
#pragma unroll
        for (int i = 0; i < ND; i++) d[wv * WSL + 64 * i + lane] = reg[i];
    };
    /* Sums in two levels, so that rounding grows with the square root of K's parts: bf16, the
     * matrix instructions of SEG stages start from zero (seg) and their sum goes onto acc; fp32,
     * four chains of two instructions a stage, summed as a tree. (One chain over a wave's whole
     * share: 3.2e-7 of the result's norm at 7168 columns in bf16 and 5.4e-7 in fp32, against
     * 2.0e-7 for a vector-unit GEMV's 112 sums per lane; so: 1.3e-7 and 1.3e-7.) */
    constexpr int SEG = ST == 3 ? 3 : 2;
    const k3_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    k3_f32x4 acc[MT][NB], seg[BF ? MT : 1][BF ? NB : 1];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int b = 0; b < NB; b++) acc[m][b] = zero;
    /* the slots of this lane's pieces in row tile 0 and token block 0 */
    constexpr int NPW = BF ? 1 : 2;
    int iw[MX ? 4 : NPW], ix[2], il[2];
    if constexpr (MX) {
#pragma unroll
        for (int q = 0; q < 4; q++) iw[q] = wv * MT * 256 + (r16 * 4 + (q ^ (r16 >> 2))) * 4 + g;
    } else {
#pragma unroll
        for (int h = 0; h < NPW; h++) iw[h] = wv * WSL + r16 * PRW + ((NPW * g + h) ^ ((r16 / RLW) & (PRW - 1)));
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
        ix[h] = wv * WSL + MT * SLW + r16 * PRX + ((XT == 1 ? 4 * h + g : 2 * g + h) ^ ((r16 / RLX) & (PRX - 1)));
        /* the last block of an odd N8 holds 8 tokens: columns 8..15 read some of its slots
         * again (a result column depends on its own operand column only, and these go unused) */
        il[h] = N8 & 1 ? ix[h] - (r16 & 8) * PRX : ix[h];
    }
    auto comp = [&](auto slot, auto step) {
        constexpr int S = decltype(step)::value;       /* of the unrolled loop */
        const k3_u32x4 *d = buf(slot);
        k3_u32x4 w[MT][NPW];
#pragma unroll
        for (int m = 0; m < MT; m++) {
            if constexpr (MX) {
                const uint32_t *wd = (S >> 2) & 1 ? w1 : w0;
                uint32_t codes = wd[iw[S & 3] + m * 256], ss = (uint32_t)__builtin_amdgcn_ds_bpermute((16 * (S & 3) + r16) * 4, (int)sc[(S >> 2) & 1][m]);
                codes = ss == 255u ? 0u : codes;       /* NaN byte: the block is 0 */
                ss = ss == 255u ? 127u : ss;
                w[m][0] = __builtin_bit_cast(k3_u32x4, k3_dequant8_bf16(codes, k3_e8m0_operand(ss)));
            } else {
#pragma unroll
                for (int h = 0; h < NPW; h++) w[m][h] = d[iw[h] + m * SLW];
            }
        }
        k3_u32x4 xv[NB][2];
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int h = 0; h < 2; h++) xv[b][h] = d[(b + 1 < NB ? ix[h] : il[h]) + b * 128];
        if constexpr (BF && XT == 1) {
#pragma unroll
            for (int b = 0; b < NB; b++) {
#pragma unroll
                for (int k = 1; k >= 0; k--)
#pragma unroll
                    for (int m = 0; m < MT; m++)
                        seg[m][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(k3_bf16x8, w[m][0]),
                                                                            __builtin_bit_cast(k3_bf16x8, xv[b][k]),
                                                                            S % SEG == 0 && k == 1 ? zero : seg[m][b], 0, 0, 0);
                if (S % SEG == SEG - 1)
#pragma unroll
                    for (int m = 0; m < MT; m++) acc[m][b] += seg[m][b];
            }
        } else if constexpr (BF) {
            constexpr int NT = GLU == 2 ? 1 : 3;
            uint4 t[2][NT];
            auto terms = [&](int b, uint4 *o) {
                if constexpr (NT == 1) o[0] = tok_round(xv[b][0], xv[b][1]);
                else tok_cut(xv[b][0], xv[b][1], o[0], o[1], o[2]);
            };
            terms(0, t[0]);
#pragma unroll
            for (int b = 0; b < NB; b++) {
                if (b + 1 < NB) terms(b + 1, t[(b + 1) & 1]);
#pragma unroll
                for (int k = NT - 1; k >= 0; k--)
#pragma unroll
                    for (int m = 0; m < MT; m++)
                        seg[m][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(k3_bf16x8, w[m][0]),
                                                                            k3_as_bf16x8(t[b & 1][k]),
                                                                            S % SEG == 0 && k == NT - 1 ? zero : seg[m][b], 0, 0, 0);
                if (S % SEG == SEG - 1)
#pragma unroll
                    for (int m = 0; m < MT; m++) acc[m][b] += seg[m][b];
            }
        } else {
#pragma unroll
            for (int b = 0; b < NB; b++)
#pragma unroll
                for (int m = 0; m < MT; m++) {
                    k3_f32x4 c[4];
#pragma unroll
                    for (int e = 0; e < 2; e++)
#pragma unroll
                        for (int j = 0; j < 4; j++)
                            c[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w[m][j >> 1][2 * (j & 1) + e]),
                                                                        __uint_as_float(xv[b][j >> 1][2 * (j & 1) + e]),
                                                                        e == 0 ? zero : c[j], 0, 0, 0);
                    acc[m][b] += (c[0] + c[1]) + (c[2] + c[3]);
                }
        }
    };
    /* vmcnt at most ST - 1 stages of copies, the other counters free; and lgkmcnt drained (this
     * wave's LDS reads are in registers) */
    constexpr int NW = ND * (ST - 1);
    constexpr int WAIT_STAGE = (NW & 15) | (7 << 4) | (15 << 8) | ((NW >> 4) << 14);
    constexpr int WAIT_LDS = 15 | (7 << 4) | (3 << 14);
    /* MX: the chunk copies lie between stage copies, so a stage's wait lets fewer stages be in
     * flight, never more; a chunk's were issued before its first stage's. */
    constexpr int UN = MX ? 8 : ST;                /* stages per loop */
    if constexpr (XT == 2) {
        fetch(s0);
        for (int s = s0; s < s1; s += UN)
            k3_tok_for<UN>([&](auto st) {
                constexpr int S = decltype(st)::value;
                stash(std::integral_constant<int, S % ST>{});
                fetch(s + S + 1);
                comp(std::integral_constant<int, S % ST>{}, st);
            });
    } else {
    if constexpr (MX) copy_w(s0 / 4, std::integral_constant<int, 0>{});
    k3_tok_for<ST - 1>([&](auto sl) { copy(s0 + decltype(sl)::value, sl); });
    for (int s = s0; s < s1; s += UN)              /* a stage past the share multiplies zeros */
        k3_tok_for<UN>([&](auto st) {
            constexpr int S = decltype(st)::value;
            __builtin_amdgcn_s_waitcnt(WAIT_LDS);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (MX && S % 4 == 0) copy_w((s + S) / 4 + 1, std::integral_constant<int, (S / 4 + 1) & 1>{});
            copy(s + S + ST - 1, std::integral_constant<int, (S + ST - 1) % ST>{});
            __builtin_amdgcn_s_waitcnt(WAIT_STAGE);
            __builtin_amdgcn_sched_barrier(0);
            comp(std::integral_constant<int, S % ST>{}, st);
        });
    }
    /* the waves' sums, in wave order */
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    k3_f32x4 *red = reinterpret_cast<k3_f32x4 *>(b0);
    if (wv > 0)
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int b = 0; b < NB; b++) red[((wv - 1) * MT * NB + m * NB + b) * 64 + lane] = acc[m][b];
    __syncthreads();
    if (wv > 0) return;
    const bool vec = ((a.ldy | a.out) & 3) == 0 && ((uintptr_t)a.y & 15) == 0;
    bool nan = false;
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int b = 0; b < NB; b++) {
#pragma unroll
            for (int k = 0; k < KW - 1; k++) acc[m][b] += red[(k * MT * NB + m * NB + b) * 64 + lane];
#pragma unroll
            for (int e = 0; e < 4; e++) nan |= acc[m][b][e] != acc[m][b][e];
        }
    if constexpr (!MX && XT != 1 && GLU != 2) {        /* (one term has no such case) */
        if (__ballot(nan)) {
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int b = 0; b < NB; b++) red[(m * NB + b) * 64 + lane] = acc[m][b];
            tok_recompute<BF>(red, (const char *)a.W + row0 * wrow, GLU ? (const char *)a.W2 + row0 * wrow : nullptr, wrow,
                              a.x + (size_t)tok0 * a.in, a.in, nrow, ntok, MT, NB);
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int b = 0; b < NB; b++) acc[m][b] = red[(m * NB + b) * 64 + lane];
        }
    }
#pragma unroll
    for (int m = 0; m < (GLU ? 1 : MT); m++)
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const int t = tok0 + 16 * b + r16, lr = 16 * m + 4 * g, r = row0 + lr;
            k3_f32x4 v = acc[m][b];
            if (t >= a.ntok || 16 * b + r16 >= 8 * N8 || lr >= nrow) continue;
            if constexpr (GLU)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    v[e] = k3_act_pair(v[e], acc[MT - 1][b][e], a.act, a.b1, a.b2);
                    if (GLU == 2) v[e] = k3_bf16_to_f32(k3_bf16_rne(v[e]));
                }
            float *o = a.y + (size_t)t * a.ldy + r;
            if (vec) {
                if (a.accumulate) v = *reinterpret_cast<const k3_f32x4 *>(o) + v;
                *reinterpret_cast<k3_f32x4 *>(o) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (lr + e < nrow) o[e] = a.accumulate ? o[e] + v[e] : v[e];
            }
        }
}

/* KB of a stage (MX: beside 2 MT KB of codes in two chunks), and the waves of a workgroup: eight where
 * two stages of theirs fit 160 KB of LDS, else four */
constexpr int tok_stage_kb(int wt, int mt, int n8) { return wt == TOK_MX ? n8 : mt * (wt == TOK_F32 ? 2 : 1) + n8; }
constexpr int tok_waves(int wt, int mt, int n8)
{
    return 8 * (2 * tok_stage_kb(wt, mt, n8) + (wt == TOK_MX ? 2 * mt : 0)) <= 160 ? 8 : 4;
}

template <int WT, int XT, int GLU, int MT, int N8>
int launch_tok(TokArgs a, hipStream_t st)
{
    /* up to four stages (MX: two or four) */
    constexpr int MX = WT == TOK_MX;
    constexpr int SKB = tok_stage_kb(WT, MT, N8), CKB = MX ? 2 * MT : 0, KW = tok_waves(WT, MT, N8);
    constexpr int RKB = (KW - 1) * MT * ((N8 + 1) / 2) - KW * SKB;       /* the sums beyond buffer 0 */
    constexpr int S4 = (160 - (RKB > 0 ? RKB : 0) - KW * CKB) / (KW * SKB), ST = XT == 2 ? 2 : S4 >= 4 ? 4 : MX ? 2 : S4;
    const int rows = GLU ? a.rpt : 16 * MT;
    a.ntt = (a.ntok + 8 * N8 - 1) / (8 * N8);
    a.items = (a.out + rows - 1) / rows * a.ntt;
    a.per_xcd = (a.items + K3_NXCD - 1) / K3_NXCD;
    hipLaunchKernelGGL((tok_gemm_kernel<WT, XT, GLU, MT, N8, KW, ST>), dim3((unsigned)(a.per_xcd * K3_NXCD)), dim3(64 * KW),
                       0, st, a);
    K3K_LAUNCH_CHECK("tok gemm launch");
    return 0;
}

/* Cycles for the workgroups that fall to the busiest CU: per workgroup, K columns of cutting x
 * (fp32 activations against bf16 weights), moving the operands (50 bytes per cycle, fitted) and
 * multiplying, of which the largest counts whole and the others by how far they do not overlap,
 * and the start, the filling of the stages and the adding up, 3 to 4 us. The overlap is fitted to 18
 * shapes at 8 matrices (1024 -> 512 to 12288 -> 16384) x 12 token counts (2 to 512): 0.4, and for
 * fp32 weights 0.2 where eight waves fit the LDS and 1 (none) where four do, one to a SIMD. The
 * shape taken is then, over those 96 products, on average 0.7 % (bf16; at most 10), 1 % (fp32; 11) and
 * 0.9 % (MXFP4; 15) slower than the best of the 18; with 0.4 for fp32 weights as well, 11 % (61).
 * Counting the dequantisation of MXFP4 codes changed no choice for the better. */
float tok_cost(int wt, int xt, int mt, int n8, int out, int ntok, int in, int cus)
{
    const long wgs = (long)((out + 16 * mt - 1) / (16 * mt)) * ((ntok + 8 * n8 - 1) / (8 * n8));
    const int nb = (n8 + 1) / 2;
    const bool f32 = wt == TOK_F32;
    const float cut = xt ? 0.f : wt == TOK_BF16 ? 16.f * nb * 5.5f / 64.f : 0.f;
    const float bytes = (16.f * mt * (f32 ? 4.f : wt == TOK_BF16 ? 2.f : 0.6f) + 8.f * n8 * 4) / 50.f;
    const float mfma = mt * nb * 512.f * (f32 ? 1.f / 256.f : (xt ? 2.f : 3.f) / 4096.f);
    const float over = !f32 ? 0.4f : tok_waves(wt, mt, n8) == 8 ? 0.2f : 1.f;
    float c = cut > bytes ? cut : bytes;
    if (mfma > c) c = mfma;
    c += over * (cut + bytes + mfma - c);
    return (c * in + (f32 ? 7200.f : 9600.f)) * (float)((wgs + cus - 1) / cus);
}

/* (row tiles, groups of 8 tokens); the last five are ever the cheapest for fp32 weights only */
const int TOK_SHAPES[17][2] = {{1, 1}, {1, 2}, {2, 1}, {2, 2}, {2, 4}, {3, 1}, {3, 2}, {3, 4}, {4, 1},
                               {4, 2}, {4, 4}, {4, 8}, {1, 3}, {1, 4}, {1, 5}, {1, 6}, {1, 8}};

/* The cheapest shape, and its cycles. */
int tok_pick(int wt, int xt, int out, int ntok, int in, float *cycles)
{
    int best = 0;
    for (int i = 0; i < (wt == TOK_F32 ? 17 : 12); i++) {
        const float c = tok_cost(wt, xt, TOK_SHAPES[i][0], TOK_SHAPES[i][1], out, ntok, in, k3k_cu_count());
        if (i == 0 || c < *cycles) {
            best = i;
            *cycles = c;
        }
    }
    return best;
}

template <int WT, int XT>
int dispatch_tok(const TokArgs &a, hipStream_t st)
{
    float c;
    const int best = tok_pick(WT, XT, a.out, a.ntok, a.in, &c);
    if constexpr (WT == TOK_F32) {
        switch (best) {
        case 12: return launch_tok<WT, XT, 0, 1, 3>(a, st);
        case 13: return launch_tok<WT, XT, 0, 1, 4>(a, st);
        case 14: return launch_tok<WT, XT, 0, 1, 5>(a, st);
        case 15: return launch_tok<WT, XT, 0, 1, 6>(a, st);
        case 16: return launch_tok<WT, XT, 0, 1, 8>(a, st);
        }
    }
    switch (best) {
    case 0: return launch_tok<WT, XT, 0, 1, 1>(a, st);
    case 1: return launch_tok<WT, XT, 0, 1, 2>(a, st);
    case 2: return launch_tok<WT, XT, 0, 2, 1>(a, st);
    case 3: return launch_tok<WT, XT, 0, 2, 2>(a, st);
    case 4: return launch_tok<WT, XT, 0, 2, 4>(a, st);
    case 5: return launch_tok<WT, XT, 0, 3, 1>(a, st);
    case 6: return launch_tok<WT, XT, 0, 3, 2>(a, st);
    case 7: return launch_tok<WT, XT, 0, 3, 4>(a, st);
    case 8: return launch_tok<WT, XT, 0, 4, 1>(a, st);
    case 9: return launch_tok<WT, XT, 0, 4, 2>(a, st);
    case 10: return launch_tok<WT, XT, 0, 4, 4>(a, st);
    default: return launch_tok<WT, XT, 0, 4, 8>(a, st);
    }
}

/* any K and alignment: fewer shapes. Two row tiles to a workgroup where they make fewer rounds of
 * workgroups: a round of them takes 1.2-1.3 times a round of one tile with bf16 weights (7169 -> 3584,
 * 128 tokens: 53.7 us in one round, 85.9 in two of one tile; 64 tokens 52.4 and 46.2, both one round),
 * and about twice it with fp32 weights, for which they have to halve the rounds (3585 -> 7168: 16 tokens
 * 21.5 us in one round, 24.5 in two; 200 tokens 253 in four, 225 in seven). Up to 8 tokens, where the
 * weights' bytes are what counts, two rounds are no slower than one of twice as many (2049 -> 7168, 2
 * tokens: bf16 7.7 and 8.2, fp32 13.0 and 14.8). */
template <int WT>
int dispatch_any(const TokArgs &a, hipStream_t st)
{
    const long ntt = a.ntok <= 32 ? 1 : (a.ntok + 63) / 64, cus = k3k_cu_count() > 0 ? k3k_cu_count() : 1;
    const long r1 = ((a.out + 15) / 16 * ntt + cus - 1) / cus, r2 = ((a.out + 31) / 32 * ntt + cus - 1) / cus;
    const bool two = (a.ntok > 8 || r1 > 2) && (WT == TOK_BF16 ? r2 < r1 : 2 * r2 <= r1);
    if (a.ntok <= 8) return two ? launch_tok<WT, 2, 0, 2, 1>(a, st) : launch_tok<WT, 2, 0, 1, 1>(a, st);
    if (a.ntok <= 16) return two ? launch_tok<WT, 2, 0, 2, 2>(a, st) : launch_tok<WT, 2, 0, 1, 2>(a, st);
    if (a.ntok <= 32) return two ? launch_tok<WT, 2, 0, 2, 4>(a, st) : launch_tok<WT, 2, 0, 1, 4>(a, st);
    return two ? launch_tok<WT, 2, 0, 2, 8>(a, st) : launch_tok<WT, 2, 0, 1, 8>(a, st);
}

}  // namespace

/* in % 8 == 0, x and W 16-byte aligned, and a row block's operand under 2 GiB. Up to four tokens
 * of fewer than 512 columns stay with the vector units: their waves would have one stage each
 * at most, and there is no weight stream to share (2 tokens of 256 -> 1024: 6.8 us either way). */
static int shape_ok(const void *x, const void *W, int in)
{
    return in >= 8 && in % 8 == 0 && in < (1 << 22) && (((uintptr_t)x | (uintptr_t)W) & 15) == 0;
}

/* One token stays on the vector units, where fp32 and bf16 weights of the same values give the same
 * bits, and so do up to four of short rows, whose sums are the more accurate there. */
extern "C" int k3k_tok_ok(int in, int ntok)
{
    return ntok > 1 && (ntok > 4 || in >= 512) && in >= 8 && in < (1 << 22);
}

extern "C" int k3k_tok_gemm(float *y, const float *x, const void *W, int bf16, int in, int out, int ntok, int ldy,
                            int accumulate, void *stream)
{
    if (in < 8 || in >= (1 << 22)) return k3k_fail("tok gemm shape", hipErrorInvalidValue);
    if (out <= 0) return 0;
    TokArgs a = {};
    a.y = y;
    a.x = x;
    a.W = W;
    a.in = in;
    a.out = out;
    a.ntok = ntok;
    a.ldy = ldy;
    a.accumulate = accumulate;
    if (!shape_ok(x, W, in))
        return bf16 ? dispatch_any<TOK_BF16>(a, (hipStream_t)stream) : dispatch_any<TOK_F32>(a, (hipStream_t)stream);
    return bf16 ? dispatch_tok<TOK_BF16, 0>(a, (hipStream_t)stream) : dispatch_tok<TOK_F32, 0>(a, (hipStream_t)stream);
}

extern "C" int k3k_tok_glu_ok(const void *x, const void *Wg, const void *Wu, int in)
{
    return shape_ok(x, Wg, in) && shape_ok(x, Wu, in);
}

extern "C" int k3k_tok_glu(float *y, const float *x, const uint16_t *Wg, const uint16_t *Wu, int in, int out, int ntok,
                           int act, float b1, float b2, int terms, void *stream)
{
    if (!k3k_tok_glu_ok(x, Wg, Wu, in)) return k3k_fail("tok glu shape", hipErrorInvalidValue);
    if (out <= 0) return 0;
    TokArgs a = {};
    a.y = y;
    a.x = x;
    a.W = Wg;
    a.W2 = Wu;
    a.in = in;
    a.out = a.ldy = out;
    a.ntok = ntok;
    a.act = act;
    a.b1 = b1;
    a.b2 = b2;
    /* half-filled tiles where those are still one round of workgroups (8 tokens of 7168 -> 3072, two
     * rounds of them: 37.6 us with the down product, 38.7 on the GEMMs): the weight stream, not the
     * products, is what takes the time */
    a.rpt = (out + 7) / 8 <= k3k_cu_count() ? 8 : 16;
    hipStream_t st = (hipStream_t)stream;
    if (terms == 1)
        return ntok <= 8    ? launch_tok<TOK_BF16, 0, 2, 2, 1>(a, st)
               : ntok <= 16 ? launch_tok<TOK_BF16, 0, 2, 2, 2>(a, st)
                            : launch_tok<TOK_BF16, 0, 2, 2, 4>(a, st);
    return ntok <= 8    ? launch_tok<TOK_BF16, 0, 1, 2, 1>(a, st)
           : ntok <= 16 ? launch_tok<TOK_BF16, 0, 1, 2, 2>(a, st)
                        : launch_tok<TOK_BF16, 0, 1, 2, 4>(a, st);
}

/* both terms reachable from xhi with 32-bit offsets */
static int terms_ok(const uint16_t *xhi, const uint16_t *xlo, int in, int ntok, uint32_t *lo_off)
{
    if (!xlo) xlo = xhi;                   /* one term */
    const uint64_t d = (uint64_t)((const char *)xlo - (const char *)xhi);
    if (xlo < xhi || d + (uint64_t)ntok * in * 2 >= 0x80000000u || (((uintptr_t)xhi | (uintptr_t)xlo) & 15)) return 0;
    *lo_off = (uint32_t)d;
    return 1;
}

extern "C" int k3k_tok_mx_ok(const uint16_t *xhi, const uint16_t *xlo, const void *packed, int in, int ntok)
{
    uint32_t lo;
    return ntok > 2 && in % 32 == 0 && in < (1 << 22) && ((uintptr_t)packed & 15) == 0 &&
           terms_ok(xhi, xlo, in, ntok, &lo);
}

/* Whether it is the faster kernel for three tokens and more. The streaming kernel (k3_mx.hip), whose
 * workgroups are tiles of 16 rows x 16 tokens with a wave per four steps of 128 columns, is it where K is
 * short, since a wave here takes at least 128 columns of K and the others idle. Two terms: up to 512
 * columns, and up to 1152 where its tiles are about one to five per CU (168 tokens of 416 -> 630 6.8 us
 * there and 9.6 here; 11 of 864 -> 7633 7.0 and 9.8; 29 of 768 -> 14889, 7 per CU, 17.1 and 13.0). One
 * term, for which it does half the work and this kernel the same: wherever its tiles' steps past the
 * seventh, 330 cycles each on a CU, are cheaper than the launch here (179 tokens of 416 -> 5503 13.3 and
 * 27.3; 172 of 1728 -> 2790 20.4 and 23.3; 144 of 7424 -> 2943 73.6 and 34.6). Over 900 products the one
 * taken is on average 0.8 % (two terms, at most 14) and 2.3 % (one, at most 26) slower than the faster one. */
extern "C" int k3k_tok_mx_pays(int in, int out, int ntok, int terms)
{
    const long tiles = (long)((out + 15) / 16) * ((ntok + 15) / 16), cus = k3k_cu_count() > 0 ? k3k_cu_count() : 1;
    if (terms == 2) return in > 512 && (in > 1152 || 5 * tiles < 4 * cus || tiles > 5 * cus);
    float c;
    tok_pick(TOK_MX, 1, out, ntok, in, &c);
    return 330.f * (float)tiles * (float)((in + 127) / 128 - 7) >= c * (float)cus;
}

extern "C" int k3k_tok_mx(float *y, const uint16_t *xhi, const uint16_t *xlo, const void *packed, const uint8_t *scales,
                          int in, int out, int ntok, int ldy, void *stream)
{
    if (!k3k_tok_mx_ok(xhi, xlo, packed, in, ntok)) return k3k_fail("tok mx shape", hipErrorInvalidValue);
    if (out <= 0) return 0;
    TokArgs a = {};
    a.y = y;
    a.xhi = xhi;
    (void)terms_ok(xhi, xlo, in, ntok, &a.lo_off);
    a.W = packed;
    a.scales = scales;
    a.in = in;
    a.out = out;
    a.ntok = ntok;
    a.ldy = ldy;
    return dispatch_tok<TOK_MX, 1>(a, (hipStream_t)stream);
}

extern "C" int k3k_tok_terms_ok(const uint16_t *xhi, const uint16_t *xlo, const uint16_t *W, int in, int ntok)
{
    uint32_t lo;
    return shape_ok(W, W, in) && terms_ok(xhi, xlo, in, ntok, &lo);
}

extern "C" int k3k_tok_terms(float *y, int ldy, int accumulate, const uint16_t *W, const uint16_t *xhi, const uint16_t *xlo,
                             int in, int out, int ntok, void *stream)
{
    if (!k3k_tok_terms_ok(xhi, xlo, W, in, ntok)) return k3k_fail("tok terms shape", hipErrorInvalidValue);
    if (out <= 0) return 0;
    TokArgs a = {};
    a.y = y;
    a.xhi = xhi;
    (void)terms_ok(xhi, xlo, in, ntok, &a.lo_off);
    a.W = W;
    a.in = in;
    a.out = out;
    a.ntok = ntok;
    a.ldy = ldy;
    a.accumulate = accumulate;
    return dispatch_tok<TOK_BF16, 1>(a, (hipStream_t)stream);
}
