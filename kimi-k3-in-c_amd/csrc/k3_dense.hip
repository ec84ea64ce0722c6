/* SPDX-License-Identifier: Apache-2.0 */
/*
 * k3_dense.hip -- dense GEMV on the vector units: fp32, bf16 and per-row int8 weights.
 *
 * Replaces k3_matmul (src/core/k3_ops.c:265-291), k3_matmul_bf16 (:1108-1213) and
 * k3_matmul_q8 (:1221-1289) of the reference for the decode shapes.
 *
 * gemv_rows_kernel (one token, and several where their rows are few; ANY: any row length and
 * alignment): a wave owns RW rows and NT tokens; lane l takes the 8-element chunks l, l+64, l+128,
 * ... of every row, and issues the loads of U chunks of all RW rows (and the matching x chunks)
 * before any arithmetic, so a lane keeps U*RW 16-byte weight loads in flight and each x chunk it
 * loads serves RW rows. Per lane the products are accumulated in fp32 in ascending column
 * order (several tokens: the 8 products of a chunk first, then their sum onto the lane's, which takes
 * the error against 64 bits from 2.0e-7 to below 1e-7), then the wave reduces with a butterfly. The
 * fp32 and bf16 kernels are one template, so on weights that are the same values they perform the same
 * operations in the same order and agree bit for bit (the reference holds the same property between its
 * two kernels, tests/unit/test_ops.c:798-848), for one token of any row length. Accumulation
 * is fp32 where the reference uses fp64; the difference is far inside max|err| <= 1e-4
 * ||ref||inf. More tokens go to the matrix cores (k3_tok.hip; two tokens of 7168 -> 3584 in
 * bf16: 13.0 us here, 10.3 there) past few_rows: there the two types are cut and summed differently and
 * agree within rounding only, and a token's sums depend on how many come with it.
 */
#include "k3_common.h"
#include "k3k.h"

namespace {

/* Draft-model int8 rows [f32 scale][int8 x in] (reference k3_ops.c:1221-1289): fp32
 * accumulation, scale applied once at the end. No exactness contract, as there. */
__global__ __launch_bounds__(256) void gemv_q8_kernel(float *y, const float *x, const uint8_t *W,
                                                      int in, int out, int ldy)
{
    const int lane = threadIdx.x & 63;
    const int o = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int t = blockIdx.y;
    if (o >= out) return;
    const uint8_t *row = W + (size_t)o * (4 + (size_t)in);
    const float *xt = x + (size_t)t * in;
    float acc = 0.0f;
    for (int i = lane; i < in; i += 64) acc = fmaf((float)(int8_t)row[4 + i], xt[i], acc);
    for (int s = 32; s > 0; s >>= 1) acc += __shfl_xor(acc, s, 64);
    if (lane == 0) {
        uint32_t u = (uint32_t)row[0] | ((uint32_t)row[1] << 8) | ((uint32_t)row[2] << 16) |
                     ((uint32_t)row[3] << 24);
        y[(size_t)t * ldy + o] = acc * __uint_as_float(u);
    }
}


/* Raw 8-element weight chunk: one 16-byte load (bf16) or two (fp32), non-temporal (NTL) where
 * aligned and streamed once per launch. */
typedef unsigned int k3u32x4 __attribute__((ext_vector_type(4)));
typedef float k3f32x4 __attribute__((ext_vector_type(4)));

typedef k3u32x4 k3u32x4_any __attribute__((aligned(2)));
typedef k3f32x4 k3f32x4_any __attribute__((aligned(4)));

template <bool ANY, bool NTL>
__device__ __forceinline__ uint4 ld16(const void *p)
{
    k3u32x4 v;
    if constexpr (ANY) v = *reinterpret_cast<const k3u32x4_any *>(p);
    else if constexpr (NTL) v = __builtin_nontemporal_load(reinterpret_cast<const k3u32x4 *>(p));
    else v = *reinterpret_cast<const k3u32x4 *>(p);
    return make_uint4(v.x, v.y, v.z, v.w);
}
template <bool ANY>
__device__ __forceinline__ float4 ldx4(const float *p)
{
    if constexpr (ANY) {
        const k3f32x4 v = *reinterpret_cast<const k3f32x4_any *>(p);
        return make_float4(v.x, v.y, v.z, v.w);
    } else {
        return *reinterpret_cast<const float4 *>(p);
    }
}
/* the first n (< 8) elements at p, zeros behind them */
template <typename T>
__device__ __forceinline__ void ld_tail(T (&v)[8], const T *p, int n)
{
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = k < n ? p[k] : T(0);
}

template <typename WT> struct Chunk8;
template <> struct Chunk8<uint16_t> {
    uint4 v;
    template <bool ANY, bool NTL>
    __device__ __forceinline__ void load(const uint16_t *p) { v = ld16<ANY, NTL>(p); }
    __device__ __forceinline__ void tail(const uint16_t *p, int n)
    {
        uint16_t t[8];
        ld_tail(t, p, n);
        v = make_uint4(t[0] | (uint32_t)t[1] << 16, t[2] | (uint32_t)t[3] << 16, t[4] | (uint32_t)t[5] << 16, t[6] | (uint32_t)t[7] << 16);
    }
    __device__ __forceinline__ float at(int k) const
    {
        const uint32_t u = k < 2 ? v.x : k < 4 ? v.y : k < 6 ? v.z : v.w;
        return __uint_as_float((k & 1) ? (u & 0xFFFF0000u) : (u << 16));
    }
};
template <> struct Chunk8<float> {
    float4 a, b;
    __device__ __forceinline__ void tail(const float *p, int n)
    {
        float t[8];
        ld_tail(t, p, n);
        a = make_float4(t[0], t[1], t[2], t[3]);
        b = make_float4(t[4], t[5], t[6], t[7]);
    }
    template <bool ANY, bool NTL>
    __device__ __forceinline__ void load(const float *p)
    {
        const uint4 u = ld16<ANY, NTL>(p), v = ld16<ANY, NTL>(p + 4);
        a = make_float4(__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z), __uint_as_float(u.w));
        b = make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w));
    }
    __device__ __forceinline__ float at(int k) const
    {
        return k == 0 ? a.x : k == 1 ? a.y : k == 2 ? a.z : k == 3 ? a.w
             : k == 4 ? b.x : k == 5 ? b.y : k == 6 ? b.z : b.w;
    }
};

template <typename WT, int RW, int NT, int U, bool ANY>
__global__ __launch_bounds__(256) void gemv_rows_kernel(float *__restrict__ y, const float *__restrict__ x,
                                                        const WT *__restrict__ W, int in, int out, int ntok, int ldy)
{
    /* (several tokens' weights are read once per NT of them: through the caches) */
    constexpr bool NTL = !ANY && NT == 1;
    const int lane = threadIdx.x & 63;
    const int r0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * RW, t0 = blockIdx.y * NT;
    if (r0 >= out) return;
    const int nch = ANY ? (in + 7) >> 3 : in >> 3;
    const WT *row[RW];
#pragma unroll
    for (int r = 0; r < RW; r++) row[r] = W + (size_t)min(r0 + r, out - 1) * in;
    const float *xt[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) xt[t] = x + (size_t)min(t0 + t, ntok - 1) * in;
    float acc[RW][NT];
#pragma unroll
    for (int r = 0; r < RW; r++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[r][t] = 0.0f;
    for (int cb = lane; cb < nch; cb += 64 * U) {
        Chunk8<WT> w[U][RW];
        float4 xa[U][NT], xb[U][NT];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int c = cb + 64 * u;
            if (ANY ? 8 * (c + 1) <= in : c < nch) {
#pragma unroll
                for (int r = 0; r < RW; r++) w[u][r].template load<ANY, NTL>(row[r] + 8 * (size_t)c);
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    xa[u][t] = ldx4<ANY>(xt[t] + 8 * (size_t)c);
                    xb[u][t] = ldx4<ANY>(xt[t] + 8 * (size_t)c + 4);
                }
            } else if (ANY && c < nch) {           /* the row's last in % 8 */
#pragma unroll
                for (int r = 0; r < RW; r++) w[u][r].tail(row[r] + 8 * (size_t)c, in - 8 * c);
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    float v[8];
                    ld_tail(v, xt[t] + 8 * (size_t)c, in - 8 * c);
                    xa[u][t] = make_float4(v[0], v[1], v[2], v[3]);
                    xb[u][t] = make_float4(v[4], v[5], v[6], v[7]);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (cb + 64 * u < nch) {
#pragma unroll
                for (int r = 0; r < RW; r++)
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        float a = NT == 1 ? acc[r][t] : 0.0f;
                        a = fmaf(w[u][r].at(0), xa[u][t].x, a);
                        a = fmaf(w[u][r].at(1), xa[u][t].y, a);
                        a = fmaf(w[u][r].at(2), xa[u][t].z, a);
                        a = fmaf(w[u][r].at(3), xa[u][t].w, a);
                        a = fmaf(w[u][r].at(4), xb[u][t].x, a);
                        a = fmaf(w[u][r].at(5), xb[u][t].y, a);
                        a = fmaf(w[u][r].at(6), xb[u][t].z, a);
                        a = fmaf(w[u][r].at(7), xb[u][t].w, a);
                        acc[r][t] = NT == 1 ? a : acc[r][t] + a;
                    }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < RW; r++)
#pragma unroll
        for (int t = 0; t < NT; t++) {
            float a = acc[r][t];
            for (int s = 32; s > 0; s >>= 1) a += __shfl_xor(a, s, 64);
            acc[r][t] = a;
        }
    if (lane == 0) {
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int r = 0; r < RW; r++)
                if (t0 + t < ntok && r0 + r < out) y[(size_t)(t0 + t) * ldy + r0 + r] = acc[r][t];
    }
}

/* gate, up and the activation of one token: a wave takes row o of both matrices, with
 * gemv_rows_kernel's sums (the same bits), and lane 0 stores act(gate, up). One launch for
 * three: the shared expert of k3_moe's one token, 2 x 88 MB, 15.9 + 15.2 + 4.5 us as two GEMVs and
 * the activation. */
template <typename WT, int U>
__global__ __launch_bounds__(256) void gemv_glu_kernel(float *__restrict__ y, const float *__restrict__ x,
                                                       const WT *__restrict__ Wg, const WT *__restrict__ Wu, int in,
                                                       int out, int act, float b1, float b2)
{
    const int lane = threadIdx.x & 63;
    const int o = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (o >= out) return;
    const int nch = in >> 3;
    const WT *row[2] = {Wg + (size_t)o * in, Wu + (size_t)o * in};
    float acc[2] = {0.0f, 0.0f};
    for (int cb = lane; cb < nch; cb += 64 * U) {
        Chunk8<WT> w[U][2];
        float4 xa[U], xb[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int c = cb + 64 * u;
            if (c < nch) {
#pragma unroll
                for (int r = 0; r < 2; r++) w[u][r].template load<false, true>(row[r] + 8 * (size_t)c);
                xa[u] = reinterpret_cast<const float4 *>(x + 8 * (size_t)c)[0];
                xb[u] = reinterpret_cast<const float4 *>(x + 8 * (size_t)c)[1];
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++)
            if (cb + 64 * u < nch) {
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    float a = acc[r];
                    a = fmaf(w[u][r].at(0), xa[u].x, a);
                    a = fmaf(w[u][r].at(1), xa[u].y, a);
                    a = fmaf(w[u][r].at(2), xa[u].z, a);
                    a = fmaf(w[u][r].at(3), xa[u].w, a);
                    a = fmaf(w[u][r].at(4), xb[u].x, a);
                    a = fmaf(w[u][r].at(5), xb[u].y, a);
                    a = fmaf(w[u][r].at(6), xb[u].z, a);
                    a = fmaf(w[u][r].at(7), xb[u].w, a);
                    acc[r] = a;
                }
            }
    }
#pragma unroll
    for (int r = 0; r < 2; r++)
        for (int s = 32; s > 0; s >>= 1) acc[r] += __shfl_xor(acc[r], s, 64);
    if (lane == 0) y[o] = k3_act_pair(acc[0], acc[1], act, b1, b2);
}

/* Launch shape of the row kernel, measured at 12288 x 7168 bf16: 2 rows per wave with 8 chunks
 * of each in flight and non-temporal weight loads stream at 6.4 TB/s (4 rows x 4 chunks with
 * cached loads: 5.6 TB/s). */
constexpr int GV_RW = 2;

/* One token of a row length that is no multiple of 8, or operands that are not 16-byte aligned: the
 * same loads at the elements they start at, through the caches, since neighbouring lanes share lines
 * (7169 -> 3584 in bf16 11.0 us, fp32 16.7; non-temporal 13.0 and 24.0; the several-token kernel 15.1
 * and 20.4; a wave per row, one load after the other, 74.9 and 99.2). */
template <typename WT, int NT, int U>
void launch_rows(float *y, const float *x, const WT *W, int in, int out, int ntok, int ldy, bool vec, hipStream_t st)
{
    const dim3 grid((unsigned)((out + 4 * GV_RW - 1) / (4 * GV_RW)), (unsigned)((ntok + NT - 1) / NT));
    if (vec) hipLaunchKernelGGL((gemv_rows_kernel<WT, GV_RW, NT, U, false>), grid, dim3(256), 0, st, y, x, W, in, out, ntok, ldy);
    else hipLaunchKernelGGL((gemv_rows_kernel<WT, GV_RW, NT, U, true>), grid, dim3(256), 0, st, y, x, W, in, out, ntok, ldy);
}

template <typename WT>
void launch_gemv(float *y, const float *x, const WT *W, int in, int out, int ntok, int ldy, bool vec, hipStream_t st)
{
    if (ntok == 1) launch_rows<WT, 1, 8>(y, x, W, in, out, ntok, ldy, vec, st);
    else if (ntok == 2) launch_rows<WT, 2, 4>(y, x, W, in, out, ntok, ldy, vec, st);
    else launch_rows<WT, 4, 2>(y, x, W, in, out, ntok, ldy, vec, st);
}

/* Several tokens stay with the rows kernel where its workgroups, of 8 rows and 4 tokens, are at most
 * one per CU (two for two tokens; four for rows at any alignment, in bf16 past 16 tokens). So small a product is the chain of a
 * wave's loads: here a wave has 8 KB of weights on their way and there is a wave per two rows, where
 * k3_tok.hip's tiles of 16 rows leave most CUs without any (bf16: 2 tokens of 7112 -> 947 6.1 us, 8.9
 * there; 43 of 6112 -> 152, 209 workgroups, 6.8 and 8.2; fp32: 2 of 8912 -> 293 8.0 and 15.2; 5 of 2208 ->
 * 921, 232, 4.9 and 7.1; 56 of 2065 -> 221, any alignment, 392, 7.9 and 21.8). Past it the CUs read rows
 * and x again and again (bf16, 5 of 9960 -> 1176, 294, 15.3 and 11.7; fp32, 58 of 9008 -> 211, 405, 21.2
 * and 15.7) -- short rows of fp32 weights excepted, whose tiles cost more to start (65 tokens of 360 -> 222,
 * 476, 3.8 and 4.5; and bf16 rows at any alignment: 7 of 5549 -> 2506, 628, 18.1 and 9.5). Over 400
 * products of 2 to 250 tokens the one taken is on average 0.7 % slower than the faster one. */
bool few_rows(int in, int out, int ntok, bool vec, bool f32)
{
    const long wgs = (long)((out + 4 * GV_RW - 1) / (4 * GV_RW)) * ((ntok + 3) / 4), cus = k3k_cu_count();
    return wgs <= cus * (!vec && (f32 || ntok > 16) ? 4 : ntok == 2 ? 2 : 1) || (f32 && vec && wgs * (in < 512 ? 512 : in) <= 2048 * cus);
}

bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

}  // namespace

extern "C" int k3k_gemv_f32(float *y, const float *x, const float *W, int in, int out, int ntok,
                            int ldy, void *stream)
{
    if (out <= 0 || ntok <= 0) return 0;
    const bool vec = in % 8 == 0 && aligned16(x) && aligned16(W);
    if (k3k_tok_ok(in, ntok) && !few_rows(in, out, ntok, vec, true)) return k3k_tok_gemm(y, x, W, 0, in, out, ntok, ldy, 0, stream);
    launch_gemv<float>(y, x, W, in, out, ntok, ldy, vec, (hipStream_t)stream);
    K3K_LAUNCH_CHECK("gemv_f32 launch");
    return 0;
}

extern "C" int k3k_gemv_bf16(float *y, const float *x, const uint16_t *W, int in, int out,
                             int ntok, int ldy, void *stream)
{
    if (out <= 0 || ntok <= 0) return 0;
    const bool vec = in % 8 == 0 && aligned16(x) && aligned16(W);
    if (k3k_tok_ok(in, ntok) && !few_rows(in, out, ntok, vec, false)) return k3k_tok_gemm(y, x, W, 1, in, out, ntok, ldy, 0, stream);
    launch_gemv<uint16_t>(y, x, W, in, out, ntok, ldy, vec, (hipStream_t)stream);
    K3K_LAUNCH_CHECK("gemv_bf16 launch");
    return 0;
}

extern "C" int k3k_gemv_glu(float *y, const float *x, const void *Wg, const void *Wu, int bf16, int in, int out, int act,
                            float b1, float b2, void *stream)
{
    if (out <= 0) return 0;
    if (in <= 0 || in % 8 || !aligned16(x) || !aligned16(Wg) || !aligned16(Wu))
        return k3k_fail("gemv_glu shape", hipErrorInvalidValue);
    const dim3 grid((unsigned)((out + 3) / 4));
    if (bf16)
        hipLaunchKernelGGL((gemv_glu_kernel<uint16_t, 8>), grid, dim3(256), 0, (hipStream_t)stream, y, x,
                           (const uint16_t *)Wg, (const uint16_t *)Wu, in, out, act, b1, b2);
    else
        hipLaunchKernelGGL((gemv_glu_kernel<float, 8>), grid, dim3(256), 0, (hipStream_t)stream, y, x, (const float *)Wg,
                           (const float *)Wu, in, out, act, b1, b2);
    K3K_LAUNCH_CHECK("gemv_glu launch");
    return 0;
}

extern "C" int k3k_gemv_q8(float *y, const float *x, const void *W, int in, int out, int ntok,
                           int ldy, void *stream)
{
    if (out <= 0 || ntok <= 0) return 0;
    hipLaunchKernelGGL(gemv_q8_kernel, dim3((out + 3) / 4, ntok), dim3(256), 0,
                       (hipStream_t)stream, y, x, (const uint8_t *)W, in, out, ldy);
    K3K_LAUNCH_CHECK("gemv_q8 launch");
    return 0;
}
