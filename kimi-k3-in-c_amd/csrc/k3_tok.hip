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
 * / 17.6 / - / 38 / 179).
 *
 *   bf16 weights: x is cut into three bf16 terms by truncation, x = h + m + l. Each cut
 *     keeps the next 8 significand bits, so the three terms hold all 24 and every product
 *     with a weight is exact; v_mfma_f32_16x16x32_bf16 adds the three into one fp32 sum.
 *     (Two rounded terms, as the expert kernels use, would lose 7 bits.) bf16 ends at 2^-133,
 *     so bits of x below that are dropped: only an |x| under 2^-109 has any.
 *   fp32 weights: v_mfma_f32_16x16x4_f32 on the values as they are.
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
 * What bounds it: for few tokens the weight stream; from about 16 tokens the reads of x, which
 * reach about 50 bytes a cycle and CU (64 is the L1's width); past that cutting x (5.5 vector
 * instructions per element: cutting with v_dot2_f32_bf16, 3.5 instructions, changed nothing)
 * and, for fp32 weights, the fp32 matrix rate (1/16 of bf16). The launch rule (tok_cost)
 * weighs these.
 *
 * Infinities and NaN: the cut of an infinite x, or a zero term against an infinite weight,
 * gives NaN where the product of the uncut values is infinite. Finite operands give none, so
 * a NaN in the sum is the sign of such a case, and that element is recomputed with plain
 * FMAs.
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

struct TokArgs {
    float *y;
    const float *x;
    const void *W;
    int in, out, ntok, ldy;
    int ntt, items, per_xcd;              /* token blocks, workgroups with work, per XCD */
};

/* the plain product of one output (the NaN case) */
template <int BF>
__device__ __noinline__ float tok_plain_dot(const void *W, const float *x, size_t row, int in)
{
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < in; k += 4)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const size_t i = row * (size_t)in + k + e;
            const float w = BF ? k3_bf16_to_f32(((const uint16_t *)W)[i]) : ((const float *)W)[i];
            s[e] = fmaf(w, x[k + e], s[e]);
        }
    return (s[0] + s[1]) + (s[2] + s[3]);
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

/* BF: bf16 weights, else fp32. Stages of 32 columns. */
template <int BF, int MT, int N8, int KW, int ST>
__global__ __launch_bounds__(64 * KW) void tok_gemm_kernel(TokArgs a)
{
    constexpr int NB = (N8 + 1) / 2;               /* matrix column blocks of 16 tokens */
    constexpr int ES = BF ? 2 : 4;                 /* bytes per weight */
    constexpr int PRW = 2 * ES, PRX = 8;           /* 16-byte pieces per row and stage */
    constexpr int RLW = 16 / PRW, RLX = 2;         /* rows to 256 bytes of LDS */
    constexpr int SLW = 16 * PRW;                  /* slots per row tile (64 per token group) */
    constexpr int WSL = MT * SLW + N8 * 64;        /* slots per wave and stage */
    constexpr int ND = WSL / 64;                   /* copy instructions per wave and stage */
    constexpr uint32_t OOB = 0x80000000u;
    static_assert(ST >= 2 && ST <= 4 && ND * (ST - 1) < 64, "stages, vmcnt field");
    static_assert((KW - 1) * MT * NB * 64 <= KW * WSL, "the sums fit stage array 0");
    /* an array per stage of a plain vector type, read at one integer index: the compiler then
     * tells a copy into one array from reads of another (through longer pointer chains it does
     * not, and waits for every copy in flight before each read) */
    __shared__ __attribute__((aligned(1024))) k3_u32x4 b0[KW * WSL], b1[KW * WSL];
    __shared__ __attribute__((aligned(1024))) k3_u32x4 b2[ST > 2 ? KW * WSL : 1], b3[ST > 3 ? KW * WSL : 1];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int item = (blockIdx.x % K3_NXCD) * a.per_xcd + (int)blockIdx.x / K3_NXCD;
    if (item >= a.items) return;
    const int tb = item % a.ntt, rb = item / a.ntt;
    const int row0 = rb * 16 * MT, tok0 = tb * 8 * N8;
    const int nrow = min(a.out - row0, 16 * MT), ntok = min(a.ntok - tok0, 8 * N8);
    const k3_rsrc rw = k3_make_rsrc((const char *)a.W + (size_t)row0 * a.in * ES, (uint32_t)nrow * (uint32_t)a.in * ES);
    const k3_rsrc rx = k3_make_rsrc(a.x + (size_t)tok0 * a.in, (uint32_t)ntok * (uint32_t)a.in * 4u);
    const int nst = (a.in + 31) / 32;
    const int s0 = wv * nst / KW, s1 = (wv + 1) * nst / KW;
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
        voff[i] = row < (isw ? nrow : ntok) ? (uint32_t)row * (uint32_t)a.in * (isw ? ES : 4) + 16u * p : OOB;
        col[i] = p * (isw ? 16 / ES : 4);
    }
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
            const bool isw = i < MT * SLW / 64;
            k3_dma16(isw ? rw : rx, &d[wv * WSL + 64 * i], col[i] < left ? voff[i] : OOB, ss * (32u * (isw ? ES : 4)));
        }
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
    int iw[NPW], ix[2], il[2];
#pragma unroll
    for (int h = 0; h < NPW; h++) iw[h] = wv * WSL + r16 * PRW + ((NPW * g + h) ^ ((r16 / RLW) & (PRW - 1)));
#pragma unroll
    for (int h = 0; h < 2; h++) {
        ix[h] = wv * WSL + MT * SLW + r16 * PRX + ((2 * g + h) ^ ((r16 / RLX) & (PRX - 1)));
        /* the last block of an odd N8 holds 8 tokens: columns 8..15 read some of its slots
         * again (a result column depends on its own operand column only, and these go unused) */
        il[h] = N8 & 1 ? ix[h] - (r16 & 8) * PRX : ix[h];
    }
    auto comp = [&](auto slot) {
        constexpr int S = decltype(slot)::value;
        const k3_u32x4 *d = buf(slot);
        k3_u32x4 w[MT][NPW];
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int h = 0; h < NPW; h++) w[m][h] = d[iw[h] + m * SLW];
        k3_u32x4 xv[NB][2];
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int h = 0; h < 2; h++) xv[b][h] = d[(b + 1 < NB ? ix[h] : il[h]) + b * 128];
        if constexpr (BF) {
            uint4 t[2][3];
            tok_cut(xv[0][0], xv[0][1], t[0][0], t[0][1], t[0][2]);
#pragma unroll
            for (int b = 0; b < NB; b++) {
                if (b + 1 < NB) tok_cut(xv[b + 1][0], xv[b + 1][1], t[(b + 1) & 1][0], t[(b + 1) & 1][1], t[(b + 1) & 1][2]);
#pragma unroll
                for (int k = 2; k >= 0; k--)
#pragma unroll
                    for (int m = 0; m < MT; m++)
                        seg[m][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(k3_bf16x8, w[m][0]),
                                                                            k3_as_bf16x8(t[b & 1][k]),
                                                                            S % SEG == 0 && k == 2 ? zero : seg[m][b], 0, 0, 0);
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
    k3_tok_for<ST - 1>([&](auto sl) { copy(s0 + decltype(sl)::value, sl); });
    for (int s = s0; s < s1; s += ST)              /* a stage past the share multiplies zeros */
        k3_tok_for<ST>([&](auto sl) {
            constexpr int S = decltype(sl)::value;
            __builtin_amdgcn_s_waitcnt(WAIT_LDS);
            __builtin_amdgcn_sched_barrier(0);
            copy(s + S + ST - 1, std::integral_constant<int, (S + ST - 1) % ST>{});
            __builtin_amdgcn_s_waitcnt(WAIT_STAGE);
            __builtin_amdgcn_sched_barrier(0);
            comp(sl);
        });
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
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int b = 0; b < NB; b++) {
            k3_f32x4 v = acc[m][b];
#pragma unroll
            for (int k = 0; k < KW - 1; k++) v += red[(k * MT * NB + m * NB + b) * 64 + lane];
            const int t = tok0 + 16 * b + r16, r = row0 + 16 * m + 4 * g;
            if (t >= a.ntok || 16 * b + r16 >= 8 * N8 || r >= a.out) continue;
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (v[e] != v[e] && r + e < a.out)
                    v[e] = tok_plain_dot<BF>(a.W, a.x + (size_t)t * a.in, (size_t)(r + e), a.in);
            float *o = a.y + (size_t)t * a.ldy + r;
            if (vec) {
                *reinterpret_cast<float4 *>(o) = make_float4(v[0], v[1], v[2], v[3]);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (r + e < a.out) o[e] = v[e];
            }
        }
}

template <int BF, int MT, int N8>
int launch_tok(TokArgs a, hipStream_t st)
{
    /* eight waves where two stages of theirs fit 160 KB of LDS, else four; up to four stages */
    constexpr int SKB = MT * (BF ? 1 : 2) + N8, KW = SKB <= 10 ? 8 : 4;
    constexpr int ST = 160 / (KW * SKB) > 4 ? 4 : 160 / (KW * SKB);
    const int nrb = (a.out + 16 * MT - 1) / (16 * MT);
    a.ntt = (a.ntok + 8 * N8 - 1) / (8 * N8);
    a.items = nrb * a.ntt;
    a.per_xcd = (a.items + K3_NXCD - 1) / K3_NXCD;
    hipLaunchKernelGGL((tok_gemm_kernel<BF, MT, N8, KW, ST>), dim3((unsigned)(a.per_xcd * K3_NXCD)), dim3(64 * KW), 0,
                       st, a);
    K3K_LAUNCH_CHECK("tok gemm launch");
    return 0;
}

/* Cycles for the workgroups that fall to the busiest CU: per workgroup, K columns of cutting x
 * (bf16), moving the operands (50 bytes per cycle) and multiplying, of which the largest counts
 * whole and the others by 0.4 (measured, how far they overlap), and about 4 us (9600 cycles) to
 * start, fill the stages and add up. */
float tok_cost(int bf, int mt, int n8, int out, int ntok, int in, int cus)
{
    const long wgs = (long)((out + 16 * mt - 1) / (16 * mt)) * ((ntok + 8 * n8 - 1) / (8 * n8));
    const int nb = (n8 + 1) / 2;
    const float cut = bf ? 16.f * nb * 5.5f / 64.f : 0.f;
    const float bytes = (16.f * mt * (bf ? 2 : 4) + 8.f * n8 * 4) / 50.f;
    const float mfma = mt * nb * 512.f * (bf ? 3.f / 4096.f : 1.f / 256.f);
    float c = cut > bytes ? cut : bytes;
    if (mfma > c) c = mfma;
    c += 0.4f * (cut + bytes + mfma - c);
    return (c * in + 9600.f) * (float)((wgs + cus - 1) / cus);
}

template <int BF>
int dispatch_tok(const TokArgs &a, hipStream_t st)
{
    static const int shapes[][2] = {{1, 1}, {1, 2}, {1, 3}, {1, 4}, {1, 5}, {1, 6}, {1, 8},
                                    {2, 1}, {2, 2}, {2, 4}, {2, 8}, {3, 1}, {3, 2}, {3, 4},
                                    {4, 1}, {4, 2}, {4, 4}, {4, 8}};
    int best = 0;
    float bc = 0;
    for (int i = 0; i < (int)(sizeof shapes / sizeof shapes[0]); i++) {
        const float c = tok_cost(BF, shapes[i][0], shapes[i][1], a.out, a.ntok, a.in, k3k_cu_count());
        if (i == 0 || c < bc) {
            best = i;
            bc = c;
        }
    }
    switch (best) {
    case 0: return launch_tok<BF, 1, 1>(a, st);
    case 1: return launch_tok<BF, 1, 2>(a, st);
    case 2: return launch_tok<BF, 1, 3>(a, st);
    case 3: return launch_tok<BF, 1, 4>(a, st);
    case 4: return launch_tok<BF, 1, 5>(a, st);
    case 5: return launch_tok<BF, 1, 6>(a, st);
    case 6: return launch_tok<BF, 1, 8>(a, st);
    case 7: return launch_tok<BF, 2, 1>(a, st);
    case 8: return launch_tok<BF, 2, 2>(a, st);
    case 9: return launch_tok<BF, 2, 4>(a, st);
    case 10: return launch_tok<BF, 2, 8>(a, st);
    case 11: return launch_tok<BF, 3, 1>(a, st);
    case 12: return launch_tok<BF, 3, 2>(a, st);
    case 13: return launch_tok<BF, 3, 4>(a, st);
    case 14: return launch_tok<BF, 4, 1>(a, st);
    case 15: return launch_tok<BF, 4, 2>(a, st);
    case 16: return launch_tok<BF, 4, 4>(a, st);
    default: return launch_tok<BF, 4, 8>(a, st);
    }
}

}  // namespace

/* in % 8 == 0, x and W 16-byte aligned, and a row block's operand under 2 GiB. Up to four tokens
 * of fewer than 512 columns stay with the vector units: their waves would have one stage each
 * at most, and there is no weight stream to share (2 tokens of 256 -> 1024: 6.8 us either way). */
extern "C" int k3k_tok_ok(const float *x, const void *W, int in, int ntok)
{
    return ntok > 1 && (ntok > 4 || in >= 512) && in >= 8 && in % 8 == 0 && in < (1 << 22) && (((uintptr_t)x | (uintptr_t)W) & 15) == 0;
}

extern "C" int k3k_tok_gemm(float *y, const float *x, const void *W, int bf16, int in, int out, int ntok, int ldy,
                            void *stream)
{
    if (!k3k_tok_ok(x, W, in, ntok)) return k3k_fail("tok gemm shape", hipErrorInvalidValue);
    if (out <= 0) return 0;
    TokArgs a = {};
    a.y = y;
    a.x = x;
    a.W = W;
    a.in = in;
    a.out = out;
    a.ntok = ntok;
    a.ldy = ldy;
    return bf16 ? dispatch_tok<1>(a, (hipStream_t)stream) : dispatch_tok<0>(a, (hipStream_t)stream);
}
