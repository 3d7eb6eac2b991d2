// Products of the stack engine (stack_kernels.h): C[m,n] = sum_k A[m,k] * W[n,k] with the layer seam in the epilogue.
//
//   bfloat16, M >= 32, K % 64 == 0: LDS-DMA staged MFMA tiles, shape by rounds x area: gemm_wide_impl.h where results leave in 16-byte pieces, otherwise
//                     gemm_glds_impl.h (v_mfma_f32_32x32x16_bf16);
//   bfloat16, other M >= 32: fp32 results as far as whole stages go by the same tiles, the rest of K by fma_tile_kernel; 16-bit results by the
//                     register-staged MFMA tiles of gemm_mfma.hip;
//   bfloat16, M <= 31: slim_kernel below - HBM-bound, the weight-streaming MFMA main loop of gemm_slim_impl.h; grouped products of many workgroups
//                     slim_group_kernel, the same with its block in registers;
//   bfloat16, M = 1:  row_kernel - dot products on the vector pipe, K split over a workgroup's waves; fp32 accumulation, DPP reduction; very many rows of
//                     one chunk: row_short_kernel (a lone token's experts: lone_up_kernel, lone_down_kernel; behind its norm: row_norm_kernel);
//   bfloat16, 2 <= M <= 8, few columns of long rows: skinny_ksplit_kernel, the same for several rows;
//   float32         : fma_tile_kernel - 64 x 64 tiles of plain fp32 FMAs through LDS (no reduced-precision matrix mode), any shape;
//                     also the fallback for bfloat16 operands whose rows are not 16-byte aligned.
//
// A row's fp32 sums run in the order of the form that serves the call, so its last bits follow the rows beside it: one row, 2 .. 31 and more are
// different orders in bfloat16, one of 2 .. 31 splits K over 2, 4 or 8 waves by its rows and by how many workgroups its launch holds
// (slim::pick_shape), one row's over 1 .. 4 by its columns and products (pick_row_shape), and a product of few tiles is cut along K by how many
// there are.  Rows of one launch do not depend on each other.
#include "dev_utils.h"
#include "gemm_glds_impl.h"
#include "gemm_seam.h"
#include "gemm_slim_impl.h"
#include "gemm_wide_impl.h"
#include "stack_kernels.h"
#include "stack_norm_impl.h"
#include "stack_route_impl.h"
#include <cmath>

namespace tllm
{
namespace kernels
{
int launch_gemm_mfma(const GemmParams& p, hipStream_t stream); // gemm_mfma.hip; 1: shape not served

using namespace dev;

namespace
{

template <int DT>
__device__ __forceinline__ float ld_el(const void* p, int64_t i)
{
    if constexpr (DT == DT_BF16)
        return bf2f(reinterpret_cast<const uint16_t*>(p)[i]);
    else
        return reinterpret_cast<const float*>(p)[i];
}

template <int DT>
__device__ __forceinline__ void seam(const StackGemmParams& p, int row, int col, float v)
{
    if (p.resid)
    {
        float g = 1.f;
        if (p.gate)
        {
            const float z = ld_el<DT>(p.gate, (int64_t) row * p.ldg + col) + (p.gate_bias ? p.gate_bias[col] : 0.f);
            g = 1.f / (1.f + expf(-z));
        }
        p.resid[(int64_t) row * p.ldr + col] += g * v;
    }
    else
    {
        if (p.bias)
            v += p.bias[col];
        seam_store<DT == DT_FLOAT>(p.seam, seam_out<DT == DT_FLOAT>(p.seam, p.act, p.c, p.ldc, p.out_f32 != 0, col), row, col, v);
    }
}

// columns col (even) and col + 1 (where it exists)
template <int DT>
__device__ __forceinline__ void seam_pair(const StackGemmParams& p, int row, int col, float v0, float v1)
{
    const bool has1 = col + 1 < p.N;
    if (p.resid)
    {
        seam<DT>(p, row, col, v0);
        if (has1)
            seam<DT>(p, row, col + 1, v1);
        return;
    }
    if (p.bias)
    {
        v0 += p.bias[col];
        v1 += has1 ? p.bias[col + 1] : 0.f;
    }
    seam_store_pair<DT == DT_FLOAT>(p.seam, p.act, p.c, p.ldc, p.out_f32 != 0, row, col, v0, v1, has1);
}

// operands of product b of a batched launch; first >= 0: of a grouped one whose rows the caller has looked up
template <int DT>
__device__ __forceinline__ StackGemmParams batch_slice(StackGemmParams p, int64_t b, int first = -1, int rows = 0)
{
    constexpr int ES = DT == DT_BF16 ? 2 : 4;
    p.a = reinterpret_cast<const char*>(p.a) + b * p.stride_a * ES;
    p.w = reinterpret_cast<const char*>(p.w) + b * p.stride_w * ES;
    if (p.c)
        p.c = reinterpret_cast<char*>(p.c) + b * p.stride_c * ((p.out_f32 || DT == DT_FLOAT) ? 4 : 2);
    if (p.group_off)
    {
        // grouped form: this product's rows are a range of a and c that the device knows
        const int64_t o = first >= 0 ? first : p.group_off[b];
        p.M = first >= 0 ? rows : p.group_off[b + 1] - (int) o;
        if (p.a_rows)
            p.a_rows += o;
        else
            p.a = reinterpret_cast<const char*>(p.a) + o * p.lda * ES;
        if (p.c)
            p.c = reinterpret_cast<char*>(p.c) + o * p.ldc * ((p.out_f32 || DT == DT_FLOAT) ? 4 : 2);
    }
    return p;
}

constexpr int TM = 64, TN = 64, TK = 16;

template <int DT>
__global__ __launch_bounds__(256) void fma_tile_kernel(const StackGemmParams p_in)
{
    const StackGemmParams p = batch_slice<DT>(p_in, blockIdx.z);
    __shared__ int64_t row_s[TM]; // where the tile's rows of a start
    __shared__ float As[TK][TM + 4];
    __shared__ float Ws[TK][TN + 4];
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
    if (m0 >= p.M)
        return; // (a group with fewer rows than the launch's bound)
    if (tid < TM)
        row_s[tid] = m0 + tid < p.M ? (int64_t) (p.a_rows ? p.a_rows[m0 + tid] : m0 + tid) * p.lda : 0;
    __syncthreads();
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            acc[i][j] = 0.f;
    for (int k0 = 0; k0 < p.K; k0 += TK)
    {
#pragma unroll
        for (int i = 0; i < 4; ++i)
        {
            const int idx = tid + i * 256, r = idx / TK, k = idx % TK;
            As[k][r] = (m0 + r < p.M && k0 + k < p.K) ? ld_el<DT>(p.a, row_s[r] + k0 + k) : 0.f;
            Ws[k][r] = (n0 + r < p.N && k0 + k < p.K) ? ld_el<DT>(p.w, (int64_t) (n0 + r) * p.ldw + k0 + k) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < TK; ++k)
        {
            float a[4], w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                a[i] = As[k][ty * 4 + i];
                w[i] = Ws[k][tx * 4 + i];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[i][j] = fmaf(a[i], w[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; j += 2)
        {
            const int row = m0 + ty * 4 + i, col = n0 + tx * 4 + j;
            if (row < p.M && col < p.N)
                seam_pair<DT>(p, row, col, acc[i][j], acc[i][j + 1]);
        }
}

// Group blockIdx.z of a grouped launch whose grid holds fewer products than there are groups: the blockIdx.z-th one that has rows (a step of
// few tokens reaches few experts; 32 x 352 workgroups of which 4 x 352 have work cost more to start than to run).  -1: there is none.
// first, rows: where its rows begin and how many they are.
__device__ __forceinline__ int nth_group(const int32_t* off, int groups, int nth, int& first, int& rows)
{
    const int lane = threadIdx.x & 63;
    for (int g0 = 0; g0 < groups; g0 += 64)
    {
        const int g = g0 + lane;
        const int lo = g < groups ? off[g] : 0, hi = g < groups ? off[g + 1] : 0;
        uint64_t has = __ballot(hi > lo);
        const int n = __popcll(has);
        if (nth < n)
        {
            for (; nth > 0; --nth)
                has &= has - 1;
            const int at = __ffsll((unsigned long long) has) - 1;
            first = __builtin_amdgcn_readlane(lo, at);
            rows = __builtin_amdgcn_readlane(hi, at) - first;
            return g0 + at;
        }
        nth -= n;
    }
    return -1;
}

// bfloat16, one row: KS waves share SK_R rows of W (one pair of columns), wave w the 1 KiB chunks w, w + KS, ... of each, and 4 / KS such teams make
// a workgroup.  NC chunks per wave and row, with the activations that face them, are requested before the first is used: a product of up to
// 512 KS NC columns of A is one trip to memory per wave, and the next workgroups' trips overlap it.  Bound by the weights' stream.  What it replaced were whole
// rows per wave, a chunk of 2 rows at a time, and for long rows of few columns the matrix pipe; us, cold weights, N x K:
//   2048 x 2048 3.5 (4.6)    2048 x 5504 6.0 (8.5)    4096 x 4096 7.0 (8.5)    4096 x 11008 16.5 (19.0)    10304 x 2048 8.0 (8.9)
//   10240 x 4096 13.6 (15.5)    22016 x 4096 26.4 = 6.8 TB/s (31.1)    32000 x 2048 20.0 (21.4); of rows below 512 bytes the new form has many a bit slower:
//   16384 x 128 5.3 (4.7)    32000 x 256 8.2 (7.4)
// These are repetitions, whose code is warm; between a step's other kernels 2048 x 2048 takes 4.6, 4096 x 4096 8.7, 10304 x 2048 10.4, 32000 x 2048 21.6.
// 4 rows per team measured the same within 4 %, 8 waves per team too, 8 of both up to 60 % worse.
constexpr int SK_R = 2;

// What the epilogue of columns n and n + 1 of the one row reads, requested with the weights; raw, so that nothing waits for it here.
struct RowSeam
{
    float r[2], b[2];
    uint16_t z[2];
};
__device__ __forceinline__ RowSeam row_seam_request(const StackGemmParams& p, int n)
{
    RowSeam o = {};
    const int n1 = n + 1 < p.N ? n + 1 : n;
    const float* bias = p.resid ? p.gate_bias : p.bias;
    if (bias)
    {
        o.b[0] = bias[n];
        o.b[1] = bias[n1];
    }
    if (p.resid)
    {
        o.r[0] = p.resid[n];
        o.r[1] = p.resid[n1];
        if (p.gate)
        {
            o.z[0] = reinterpret_cast<const uint16_t*>(p.gate)[n];
            o.z[1] = reinterpret_cast<const uint16_t*>(p.gate)[n1];
        }
    }
    return o;
}
// seam_pair of row 0 with those operands
__device__ __forceinline__ void row_seam(const StackGemmParams& p, const RowSeam& o, int n, float v0, float v1)
{
    if (!p.resid)
    {
        seam_store_pair<false>(p.seam, p.act, p.c, p.ldc, p.out_f32 != 0, 0, n, v0 + o.b[0], v1 + o.b[1], n + 1 < p.N);
        return;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
    {
        const float g = p.gate ? 1.f / (1.f + expf(-(bf2f(o.z[i]) + o.b[i]))) : 1.f;
        if (n + i < p.N)
            p.resid[n + i] = o.r[i] + g * (i ? v1 : v0);
    }
}

// SCALED: the row counts as scale times itself, rounded to bfloat16.  part: LDS
template <int KS, int NC, bool SCALED>
__device__ __forceinline__ void row_product(const StackGemmParams& p, float scale, float (&part)[4][SK_R])
{
    constexpr int TEAMS = 4 / KS;
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kw = wid % KS;
    const int n0 = (blockIdx.x * TEAMS + wid / KS) * SK_R; // (a team beyond N repeats the last row and stores nothing)
    const uint16_t* a = reinterpret_cast<const uint16_t*>(p.a) + (int64_t) (p.a_rows ? p.a_rows[0] : 0) * p.lda;
    const uint16_t* w[SK_R];
#pragma unroll
    for (int r = 0; r < SK_R; ++r)
        w[r] = reinterpret_cast<const uint16_t*>(p.w) + (int64_t) (n0 + r < p.N ? n0 + r : p.N - 1) * p.ldw;
    const RowSeam ops = row_seam_request(p, n0 < p.N ? n0 : p.N - 1);
    float acc[SK_R] = {0.f, 0.f};
    for (int c0 = kw; c0 * 512 < p.K; c0 += KS * NC)
    {
        uint4 wv[NC][SK_R], xv[NC];
#pragma unroll
        for (int i = 0; i < NC; ++i)
        {
            int k = (c0 + i * KS) * 512 + lane * 8;
            k = k < p.K ? k : 0; // (loads without a branch; what they bring beyond K is dropped below)
#pragma unroll
            for (int r = 0; r < SK_R; ++r)
                wv[i][r] = ld_nt16(w[r] + k);
            xv[i] = *reinterpret_cast<const uint4*>(a + k);
        }
#pragma unroll
        for (int i = 0; i < NC; ++i)
        {
            const bool in = (c0 + i * KS) * 512 + lane * 8 < p.K; // (no branch: behind one the compiler would request a chunk where it is used)
            uint32_t xs[4] = {in ? xv[i].x : 0u, in ? xv[i].y : 0u, in ? xv[i].z : 0u, in ? xv[i].w : 0u};
            if constexpr (SCALED)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    xs[q] = (uint32_t) f2bf(scale * __builtin_bit_cast(float, xs[q] << 16)) | ((uint32_t) f2bf(scale * __builtin_bit_cast(float, xs[q] & 0xffff0000u)) << 16);
#pragma unroll
            for (int r = 0; r < SK_R; ++r)
            {
                const uint32_t ws[4] = {in ? wv[i][r].x : 0u, in ? wv[i][r].y : 0u, in ? wv[i][r].z : 0u, in ? wv[i][r].w : 0u};
#pragma unroll
                for (int q = 0; q < 4; ++q)
                {
                    acc[r] = fmaf(__builtin_bit_cast(float, xs[q] << 16), __builtin_bit_cast(float, ws[q] << 16), acc[r]);
                    acc[r] = fmaf(__builtin_bit_cast(float, xs[q] & 0xffff0000u), __builtin_bit_cast(float, ws[q] & 0xffff0000u), acc[r]);
                }
            }
        }
    }
    static_assert(SK_R == 2, "a team's rows are one pair of columns");
    const float s0 = wave_sum(acc[0]), s1 = wave_sum(acc[1]);
    if constexpr (KS == 1)
    {
        if (lane == 0 && n0 < p.N)
            row_seam(p, ops, n0, s0, s1);
        return;
    }
    if (lane == 0)
    {
        part[wid][0] = s0;
        part[wid][1] = s1;
    }
    __syncthreads();
    if (lane == 0 && kw == 0 && n0 < p.N)
    {
        float v0 = part[wid][0], v1 = part[wid][1];
#pragma unroll
        for (int k = 1; k < KS; ++k)
        {
            v0 += part[wid + k][0];
            v1 += part[wid + k][1];
        }
        row_seam(p, ops, n0, v0, v1);
    }
}

template <int KS, int NC>
__global__ __launch_bounds__(256) void row_kernel(const StackGemmParams p_in, int groups)
{
    __shared__ float part[4][SK_R];
    int b = blockIdx.z, first = -1, rows = 0;
    if (groups && (b = nth_group(p_in.group_off, groups, b, first, rows)) < 0)
        return;
    const StackGemmParams p = batch_slice<DT_BF16>(p_in, b, first, rows);
    if (p.M > 0)
        row_product<KS, NC, false>(p, 1.f, part);
}

// Rows of W of one chunk where there are very many (a head's vocabulary on a narrow stream, the per-head products of latent attention): a wave has
// SHORT_PAIRS pairs of columns, all requested at once, and half as many workgroups come and go, which is what bounds such a launch.  us, in brackets
// row_kernel<1, 1>, whole rows by the waves in turn before that: 32000 x 64 6.8 (8.1, 7.2)    32000 x 256 6.9 (8.3, 7.4)    32000 x 512 8.2 (8.8, 8.8)
//   128 heads of 512 x 128 11.1 (14.0, 12.2)    64 of 512 x 256 6.9 (8.4, 7.5)    4 pairs: 10.2, 7.5
constexpr int SHORT_PAIRS = 2, SHORT_COLS = 4 * SK_R * SHORT_PAIRS;

__global__ __launch_bounds__(256) void row_short_kernel(const StackGemmParams p_in, int groups)
{
    int b = blockIdx.z, first = -1, rows = 0;
    if (groups && (b = nth_group(p_in.group_off, groups, b, first, rows)) < 0)
        return;
    const StackGemmParams p = batch_slice<DT_BF16>(p_in, b, first, rows);
    const int lane = threadIdx.x & 63, n0 = (blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * SK_R * SHORT_PAIRS;
    if (p.M <= 0 || n0 >= p.N)
        return;
    const uint16_t* a = reinterpret_cast<const uint16_t*>(p.a) + (int64_t) (p.a_rows ? p.a_rows[0] : 0) * p.lda;
    const bool in = lane * 8 < p.K;
    const int k = in ? lane * 8 : 0;
    uint4 wv[SK_R * SHORT_PAIRS];
#pragma unroll
    for (int r = 0; r < SK_R * SHORT_PAIRS; ++r)
        wv[r] = ld_nt16(reinterpret_cast<const uint16_t*>(p.w) + (int64_t) (n0 + r < p.N ? n0 + r : p.N - 1) * p.ldw + k);
    const uint4 xv = *reinterpret_cast<const uint4*>(a + k);
    RowSeam ops[SHORT_PAIRS];
#pragma unroll
    for (int i = 0; i < SHORT_PAIRS; ++i)
        ops[i] = row_seam_request(p, n0 + SK_R * i < p.N ? n0 + SK_R * i : p.N - 1);
    const uint32_t xs[4] = {in ? xv.x : 0u, in ? xv.y : 0u, in ? xv.z : 0u, in ? xv.w : 0u};
    float sum[SK_R * SHORT_PAIRS];
#pragma unroll
    for (int r = 0; r < SK_R * SHORT_PAIRS; ++r)
    {
        const uint32_t ws[4] = {in ? wv[r].x : 0u, in ? wv[r].y : 0u, in ? wv[r].z : 0u, in ? wv[r].w : 0u};
        float acc = 0.f;
#pragma unroll
        for (int q = 0; q < 4; ++q)
        {
            acc = fmaf(__builtin_bit_cast(float, xs[q] << 16), __builtin_bit_cast(float, ws[q] << 16), acc);
            acc = fmaf(__builtin_bit_cast(float, xs[q] & 0xffff0000u), __builtin_bit_cast(float, ws[q] & 0xffff0000u), acc);
        }
        sum[r] = wave_sum(acc);
    }
#pragma unroll
    for (int i = 0; i < SHORT_PAIRS; ++i)
        if (lane == 0 && n0 + SK_R * i < p.N)
            row_seam(p, ops[i], n0 + SK_R * i, sum[SK_R * i], sum[SK_R * i + 1]);
}

// row_kernel whose row is formed here (StackRowNorm) instead of by a launch of its own in front, which costs its start and 2.3 us for some hundred cycles of work: the
// row is requested ahead of the weights and normed while they are under way.  K <= 512 KS NC.  Rows of more than 2048 values by whole waves, 8 columns a workgroup, as
// every workgroup reads the row (10240 x 4096 by 2 columns a workgroup 21.6), but for few columns.  us in a step of one token, norm + product and here: 10304 x 2048 2.3 + 11.0, 10.5;
// 11008 x 2048 2.3 + 11.2, 11.1; 10240 x 4096, 4 parts 4.6 + 14.7, 17.5; 16384 x 4096, 4 parts 4.6 + 21.0, 24.5;
// 2048 x 4096, 8 parts 3.3 + 5.9, 7.0 (with sums in another order, of quarters of a row, 5.8; so by 4 columns a workgroup 6.5, by 2 7.3).
template <int KS, int NC, int NP, int PARTS>
__global__ __launch_bounds__(256) void row_norm_kernel(const StackGemmParams p, const StackRowNorm n)
{
    constexpr int TEAMS = 4 / KS;
    constexpr int SUMS = KS == 1 && NC > 4 ? 4 : 1; // of a wave: K in the parts, and their order, of row_kernel's waves, which share rows of more than 2048
    __shared__ __attribute__((aligned(16))) uint16_t row[NP * 1024];
    __shared__ __attribute__((aligned(16))) float red[LoneRow<NP, PARTS>::SUMS];
    __shared__ float part[4][SK_R];
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kw = wid % KS;
    const int n0 = (blockIdx.x * TEAMS + wid / KS) * SK_R;
    LoneRow<NP, PARTS> lone;
    lone.request(n, p.K);
    uint4 wv[NC][SK_R];
#pragma unroll
    for (int i = 0; i < NC; ++i)
    {
        const int k = (kw + i * KS) * 512 + lane * 8;
#pragma unroll
        for (int r = 0; r < SK_R; ++r)
            wv[i][r] = ld_nt16(reinterpret_cast<const uint16_t*>(p.w) + (int64_t) (n0 + r < p.N ? n0 + r : p.N - 1) * p.ldw + (k < p.K ? k : 0));
    }
    const RowSeam ops = row_seam_request(p, n0 < p.N ? n0 : p.N - 1);
    lone.finish(n, p.K, row, red, blockIdx.x == 0);
    float acc[SUMS][SK_R] = {};
#pragma unroll
    for (int i = 0; i < NC; ++i)
    {
        const int k = (kw + i * KS) * 512 + lane * 8;
        const bool in = k < p.K;
        const uint4 xv = *reinterpret_cast<const uint4*>(row + (in ? k : 0));
        const uint32_t xs[4] = {in ? xv.x : 0u, in ? xv.y : 0u, in ? xv.z : 0u, in ? xv.w : 0u};
#pragma unroll
        for (int r = 0; r < SK_R; ++r)
        {
            const uint32_t ws[4] = {in ? wv[i][r].x : 0u, in ? wv[i][r].y : 0u, in ? wv[i][r].z : 0u, in ? wv[i][r].w : 0u};
#pragma unroll
            for (int q = 0; q < 4; ++q)
            {
                acc[i % SUMS][r] = fmaf(__builtin_bit_cast(float, xs[q] << 16), __builtin_bit_cast(float, ws[q] << 16), acc[i % SUMS][r]);
                acc[i % SUMS][r] = fmaf(__builtin_bit_cast(float, xs[q] & 0xffff0000u), __builtin_bit_cast(float, ws[q] & 0xffff0000u), acc[i % SUMS][r]);
            }
        }
    }
    float v0 = wave_sum(acc[0][0]), v1 = wave_sum(acc[0][1]);
#pragma unroll
    for (int k = 1; k < SUMS; ++k)
    {
        v0 += wave_sum(acc[k][0]);
        v1 += wave_sum(acc[k][1]);
    }
    if constexpr (KS > 1)
    {
        if (lane == 0)
        {
            part[wid][0] = v0;
            part[wid][1] = v1;
        }
        __syncthreads();
        v0 = part[wid - kw][0], v1 = part[wid - kw][1];
#pragma unroll
        for (int k = 1; k < KS; ++k)
        {
            v0 += part[wid - kw + k][0];
            v1 += part[wid - kw + k][1];
        }
    }
    if (lane == 0 && kw == 0 && n0 < p.N)
        row_seam(p, ops, n0, v0, v1);
}

// A lone token's experts, product z = choice z.  up: every wave chooses from the logits by itself (some 0.8 us in front of its weights' requests), which
// replaces a launch that orders pairs: a last workgroup that waits for all logits, chooses, orders and copies.  Choice, order and products of
// a layer of 32 + 2 outputs, width 2048, in a step of one token: 9.5 us for the router's launch, 3.7 for its logits alone.
template <int KS, int NC>
__global__ __launch_bounds__(256) void lone_up_kernel(const StackGemmParams p_in, const StackMoeParams m)
{
    __shared__ float part[4][SK_R];
    const int lane = threadIdx.x & 63, z = blockIdx.z, o = lane < m.experts + m.identity ? lane : 0;
    const Chosen c = choose_in_wave(m, m.logits[o] + (m.bias ? m.bias[o] : 0.f), m.correction ? m.correction[o] : 0.f, lane);
    if (blockIdx.x == 0 && z == 0 && (int) threadIdx.x < m.top)
    {
        m.topk_idx[lane] = c.output;
        m.topk_w[lane] = c.weight;
        m.slot_of_pair[lane] = c.output < m.experts ? lane : -1;
    }
    const int e = __builtin_amdgcn_readlane(c.output, z);
    if (e >= m.experts)
        return;
    const float scale = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, c.weight), z));
    StackGemmParams p = p_in;
    p.w = reinterpret_cast<const uint16_t*>(p.w) + e * p.stride_w;
    p.c = reinterpret_cast<char*>(p.c) + z * p.ldc * (p.out_f32 ? 4 : 2);
    if (m.weight_input)
        row_product<KS, NC, true>(p, scale, part);
    else
        row_product<KS, NC, false>(p, 1.f, part);
}

template <int KS, int NC>
__global__ __launch_bounds__(256) void lone_down_kernel(const StackGemmParams p_in, const int32_t* choice, int experts)
{
    __shared__ float part[4][SK_R];
    const int z = blockIdx.z, e = choice[z];
    if (e >= experts)
        return;
    StackGemmParams p = p_in;
    p.a = reinterpret_cast<const uint16_t*>(p.a) + z * p.lda;
    p.w = reinterpret_cast<const uint16_t*>(p.w) + e * p.stride_w;
    p.c = reinterpret_cast<char*>(p.c) + z * p.ldc * (p.out_f32 ? 4 : 2);
    row_product<KS, NC, false>(p, 1.f, part);
}

// A wave's chunks at once are all it has up to 12288 columns of A, then portions of 3.  Rows of up to 2048 columns are shared by 2 or 4 waves only where
// that leaves the chip room to take all workgroups in at once; otherwise, and where a workgroup first looks up its group, a wave has rows of its own and a
// workgroup lives longer (32000 x 2048 21.6 us by two waves a row, 22.2 by four; 4 grouped products of 2816 x 2048 10.3 against 12.1;
// 2048 x 2048 4.8 by two, 4.6 by four).  Grouped rows of 5 and 6 chunks: by two waves of 3, by one of 6, by one in two portions, us for 4 products: 704 x
// 2304 5.5 / - / -, 1408 x 2304 7.7 / 7.4 / -, 2816 x 2304 12.3 / 12.4 / 11.5, 5504 x 2304 19.7 / 19.9 / 18.5 (by two waves of 4, as longer rows: 5.8, 8.2, 12.7, 21.1).
template <int KS_, int NC_>
struct RowShape
{
    static constexpr int KS = KS_, NC = NC_, cols = SK_R * (4 / KS_);
};
template <class F>
void pick_row_shape(int64_t n, int k, int products, bool looks_up, F f)
{
    const int chunks = (k + 511) / 512, cus = launch_util::device_cus();
    const bool many = looks_up || n * products > 16 * cus;
    if (chunks <= 1)
        f(RowShape<1, 1>());
    else if (chunks <= 2)
        many ? f(RowShape<1, 2>()) : f(RowShape<2, 1>());
    else if (chunks <= 3)
        many ? f(RowShape<1, 3>()) : f(RowShape<4, 1>());
    else if (chunks <= 4)
        many ? f(RowShape<1, 4>()) : f(RowShape<4, 1>());
    else if (chunks <= 6 && looks_up)
    {
        const int64_t rows = n * products;
        rows > 32 * cus ? f(RowShape<1, 3>()) : rows > 16 * cus ? f(RowShape<1, 6>()) : f(RowShape<2, 3>());
    }
    else if (chunks <= 8)
        looks_up ? f(RowShape<2, 4>()) : f(RowShape<4, 2>());
    else if (chunks <= 12 || chunks > 24)
        f(RowShape<4, 3>());
    else if (chunks <= 16)
        f(RowShape<4, 4>());
    else
        f(RowShape<4, 6>());
}

void launch_row(const StackGemmParams& p, int products, int groups, hipStream_t stream)
{
    // (us by row_kernel and here: 10240 x 256 4.3 and 4.6, 11008 x 256 4.7 and 4.6, 16384 x 256 5.4 and 5.0, x 512 5.6 and 5.9, 20000 x 512 7.0 and 6.5)
    if (p.K <= 512 && (int64_t) p.N * products > (p.K <= 256 ? 42 : 64) * launch_util::device_cus())
    {
        hipLaunchKernelGGL(row_short_kernel, dim3((p.N + SHORT_COLS - 1) / SHORT_COLS, 1, products), dim3(256), 0, stream, p, groups);
        return;
    }
    pick_row_shape(p.N, p.K, products, p.group_off != nullptr, [&](auto shape) {
        using S = decltype(shape);
        hipLaunchKernelGGL((row_kernel<S::KS, S::NC>), dim3((p.N + S::cols - 1) / S::cols, 1, products), dim3(256), 0, stream, p, groups);
    });
}

// bfloat16, 2 .. 31 rows: the main loop of gemm_slim_impl.h, a workgroup per S::cols columns and product
template <class S>
__global__ __launch_bounds__(S::waves * 64) void slim_kernel(const StackGemmParams p_in, int groups)
{
    extern __shared__ __attribute__((aligned(16))) char slim_lds[];
    int b = blockIdx.z, first = -1, rows = 0;
    if (groups && (b = nth_group(p_in.group_off, groups, b, first, rows)) < 0)
        return;
    const StackGemmParams p = batch_slice<DT_BF16>(p_in, b, first, rows);
    if (p.M <= 0)
        return;
    const int lane = threadIdx.x & 63, n0 = blockIdx.x * S::cols;
    slim::stream<W_BF16, S>(slim_lds, reinterpret_cast<const char*>(p.w) + (int64_t) n0 * p.ldw * 2, p.ldw * 2, p.N - n0, p.K * 2,
        [&](int m) {
            m = m < p.M ? m : p.M - 1;
            return reinterpret_cast<const char*>(p.a) + (int64_t) (p.a_rows ? p.a_rows[m] : m) * p.lda * 2;
        },
        [&](int t, const slim::f32x4& acc) {
            const int row = 16 * t + (lane & 15), c = 4 * (lane >> 4), col = n0 + c;
            if (row >= p.M || row >= S::mt * S::cols || c >= S::cols)
                return;
            if (col < p.N)
                seam_pair<DT_BF16>(p, row, col, acc[0], acc[1]);
            if (col + 2 < p.N)
                seam_pair<DT_BF16>(p, row, col + 2, acc[2], acc[3]);
        });
}

// Grouped, up to 16 * MT rows a group (groups_by_registers): the same with a block ahead in registers
template <int MT>
__global__ __launch_bounds__(256) void slim_group_kernel(const StackGemmParams p_in, int groups)
{
    __shared__ __attribute__((aligned(16))) char lds[slim::lds_bytes<MT, 4>()];
    int b = blockIdx.z, first = -1, rows = 0;
    if (groups && (b = nth_group(p_in.group_off, groups, b, first, rows)) < 0)
        return;
    const StackGemmParams p = batch_slice<DT_BF16>(p_in, b, first, rows);
    if (p.M <= 0)
        return;
    const int lane = threadIdx.x & 63, n0 = blockIdx.x * 16;
    const char* xrow[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
    {
        int m = 16 * t + (lane & 15);
        m = m < p.M ? m : p.M - 1;
        xrow[t] = reinterpret_cast<const char*>(p.a) + (int64_t) (p.a_rows ? p.a_rows[m] : m) * p.lda * 2;
    }
    slim::product<W_BF16, MT, 4>(lds, reinterpret_cast<const char*>(p.w) + (int64_t) n0 * p.ldw * 2, p.ldw * 2, p.N - n0, p.K * 2, xrow,
        [&](int t, const slim::f32x4& acc) {
            const int row = 16 * t + (lane & 15), col = n0 + 4 * (lane >> 4);
            if (row >= p.M)
                return;
            if (col < p.N)
                seam_pair<DT_BF16>(p, row, col, acc[0], acc[1]);
            if (col + 2 < p.N)
                seam_pair<DT_BF16>(p, row, col + 2, acc[2], acc[3]);
        });
}

void launch_slim(const StackGemmParams& p, int products, int groups, hipStream_t stream)
{
    if (p.group_off && slim::groups_by_registers(p.M, p.N, products, (int64_t) p.K * 2, launch_util::device_cus()))
    {
        const auto kernel = p.M <= 16 ? slim_group_kernel<1> : slim_group_kernel<2>;
        hipLaunchKernelGGL(kernel, dim3((p.N + 15) / 16, 1, products), dim3(256), 0, stream, p, groups);
        return;
    }
    slim::pick_shape(p.M, p.N, products, (int64_t) p.K * 2, p.group_off != nullptr, launch_util::device_cus(), [&](auto shape) {
        using S = decltype(shape);
        launch_util::ensure_dynamic_lds(reinterpret_cast<const void*>(&slim_kernel<S>), S::lds_bytes);
        hipLaunchKernelGGL((slim_kernel<S>), dim3((p.N + S::cols - 1) / S::cols, 1, products), dim3(S::waves * 64), S::lds_bytes, stream, p, groups);
    });
}

// Several rows through few columns (a token input's gate): a workgroup per SK_R rows of W whose 4 waves split K; their sums meet in LDS.
template <int MR>
__global__ __launch_bounds__(256) void skinny_ksplit_kernel(const StackGemmParams p)
{
    __shared__ float part[4][SK_R][MR];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int n0 = blockIdx.x * SK_R;
    float acc[SK_R][MR];
#pragma unroll
    for (int r = 0; r < SK_R; ++r)
#pragma unroll
        for (int m = 0; m < MR; ++m)
            acc[r][m] = 0.f;
    const uint16_t* a = reinterpret_cast<const uint16_t*>(p.a);
    const uint16_t* w = reinterpret_cast<const uint16_t*>(p.w);
    for (int k = (wid * 64 + lane) * 8; k < p.K; k += 256 * 8)
    {
        uint4 wv[SK_R];
#pragma unroll
        for (int r = 0; r < SK_R; ++r)
            wv[r] = n0 + r < p.N ? ld_nt16(w + (int64_t) (n0 + r) * p.ldw + k) : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int m = 0; m < MR; ++m)
        {
            if (m >= p.M)
                break;
            const uint4 xv = *reinterpret_cast<const uint4*>(a + (int64_t) m * p.lda + k);
            const uint32_t xs[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
            for (int r = 0; r < SK_R; ++r)
            {
                const uint32_t ws[4] = {wv[r].x, wv[r].y, wv[r].z, wv[r].w};
#pragma unroll
                for (int i = 0; i < 4; ++i)
                {
                    acc[r][m] = fmaf(__builtin_bit_cast(float, xs[i] << 16), __builtin_bit_cast(float, ws[i] << 16), acc[r][m]);
                    acc[r][m] = fmaf(__builtin_bit_cast(float, xs[i] & 0xffff0000u), __builtin_bit_cast(float, ws[i] & 0xffff0000u), acc[r][m]);
                }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < SK_R; ++r)
#pragma unroll
        for (int m = 0; m < MR; ++m)
        {
            const float s = wave_sum(acc[r][m]);
            if (lane == 0)
                part[wid][r][m] = s;
        }
    __syncthreads();
    const int m = threadIdx.x;
    if (m < MR && m < p.M)
        seam_pair<DT_BF16>(p, m, n0, (part[0][0][m] + part[1][0][m]) + (part[2][0][m] + part[3][0][m]),
            (part[0][1][m] + part[1][1][m]) + (part[2][1][m] + part[3][1][m]));
}

// the parts of a product cut along K: their sum, in the order of K, through the product's epilogue
__global__ __launch_bounds__(256) void split_sum_kernel(const StackGemmParams p, const float* ws, int parts)
{
    const int64_t i = (int64_t) blockIdx.x * 256 + threadIdx.x, n = (int64_t) p.M * p.N;
    if (i >= n)
        return;
    float v = 0.f;
    for (int k = 0; k < parts; ++k)
        v += ws[(int64_t) k * n + i];
    seam<DT_BF16>(p, (int) (i / p.N), (int) (i % p.N), v);
}

inline int launched(const char* what)
{
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
    {
        set_error("%s launch failed: %s", what, hipGetErrorString(e));
        return -1;
    }
    return 0;
}

// Rows of a group are expected to spread around m by its root: how many tiles of `high` rows a group has on average.
inline double expected_tiles(int m, int high)
{
    double tiles = 1.0;
    for (int at = high; at < 3 * m + 16; at += high) // one more for every group of more than `at` rows
        tiles += 0.5 * std::erfc((at - m) / std::sqrt(2.0 * m));
    return tiles;
}
// The tiles of a grouped product of gemm_wide_impl.h by what they are expected to take, us: rounds of the chip x (a tile's launch, first requests and results, and its K-tiles), or
// the weights' way from HBM (5.1 TB/s), whichever is longer, rounded off between the two.  A product by itself may be off by a third, where its random groups just do or don't make
// another round; what counts is the form.  Checked on 1639 products of 8 .. 64 groups of 40 .. 560 rows, N 704 .. 5504, K 512 .. 4096, cold weights, each with sizes spread by their root (as
// a balanced router's choices are: 120 rows +- 10) and by another eighth: they take 0.92 of the time of the forms that rounds and area picked (128 x 128, 128 x 256, lock-step 256 x 256); 2
// in 100, most of which cross from one round to the next, take over 1.03 of it.  A round of few tiles costs a whole one: counted in parts it picked no better.
// us, 128 x 256 / 256 x 256 / up to 288 x 192, 32 groups of 120 rows, 2816, 2048 94.5 / 110 / 94, of 128 111 / 116 / 95, of 160 112 / 121 / 99, of 216 121 / 122 / 107 (in a step, of 120: 102
// the first and 97 the last on one card, 107 and 108 on another); 2048, 1408 63 / 44 / 57, 62 / 46 / 57, 61 / 51 / 63, 64 / 54 / 78, of 288 89 / 98 / 97; of 256, 5504, 4096 476 / 523 / 390, 4096, 2752 272 / 295 / 216; of 375, 4224, 3072
// 392 / 400 / 338.
enum GroupForm
{
    GROUP_128x128, // up to 64 rows
    GROUP_128x256,
    GROUP_256x256,
    GROUP_TALL
};
GroupForm pick_group_form(const GemmParams& g, int m)
{
    const double kt = g.K / 64, cus = launch_util::device_cus(), weights = (double) g.batch * g.N * g.K * 2 / 5.1e6;
    auto us = [&](int high, int wide, double fixed, double k_tile) {
        const double tiles = expected_tiles(m, high) * g.batch * ((g.N + wide - 1) / wide) / cus;
        const double a = std::max(1.0, std::ceil(tiles - 0.03)) * (fixed + kt * k_tile), b = fixed + weights;
        return std::sqrt(std::sqrt(a * a * a * a + b * b * b * b));
    };
    GroupForm form = GROUP_128x256;
    double best = us(128, 256, 6.6, 0.86);
    auto offer = [&](GroupForm f, double t) {
        if (t < best)
        {
            best = t;
            form = f;
        }
    };
    if (m <= 64)
        offer(GROUP_128x128, us(128, 128, 5.5, 0.45));
    offer(GROUP_256x256, us(256, 256, 9.5, m + 1.5 * std::sqrt(m) <= 128 ? 0.95 : 1.42));
    if (wide::tall_serves(g))
        offer(GROUP_TALL, us(wide::TALL_BM, wide::TALL_BN, 7.1, 0.34 + 0.004 * std::min<double>(wide::TALL_BM, m / expected_tiles(m, wide::TALL_BM))));
    return form;
}

// The tile shapes of the LDS-DMA kernels, all with stages of whole 128-byte lines and 8 waves, and what a tile of each kind costs per area when
// the chip is full of them (measured, relative to lock-step 256 x 256; M 2048 .. 512, N 2048 .. 22016, K 2048 .. 11008): fewest workgroup rounds x
// area x cost.  row_tiles: those of 128 rows by gemm_wide_impl.h, 4 - 18 % quicker than the lock-step ones of gemm_glds_impl.h (figures there), which stay for
// what leaves in other pieces (columns that are no multiple of 8, rows off 16 bytes) and for 256 rows x 192, where the 16 x 16 form gained nothing.
int launch_glds_bf16(const GemmParams& g, hipStream_t stream, int m_expected = 0)
{
    struct Shape
    {
        int id, bm, bn;
        double f;
    };
    static const Shape lock_step[] = {{0, 128, 128, 1.49}, {1, 256, 192, 1.16}, {2, 256, 256, 1.0}, {3, 128, 256, 1.15}, {4, 128, 192, 1.28}, {5, 128, 64, 2.15}};
    static const Shape row_tiles[] = {{0, 128, 128, 1.37}, {1, 256, 192, 1.16}, {2, 256, 256, 1.0}, {3, 128, 256, 1.07}, {4, 128, 192, 1.22}, {5, 128, 64, 2.05}};
    const bool served = wide::serves<W_BF16>(g);
    const Shape (&shapes)[6] = served ? row_tiles : lock_step;
    const int cus = launch_util::device_cus();
    double best = 1e30;
    int pick = 0;
    for (const Shape& sh : shapes)
    {
        const int m = m_expected > 0 ? m_expected : g.M;
        const int64_t tiles = (int64_t) ((m + sh.bm - 1) / sh.bm) * ((g.N + sh.bn - 1) / sh.bn) * (g.batch > 1 ? g.batch : 1);
        const double cost = (double) ((tiles + cus - 1) / cus) * sh.bm * sh.bn * sh.f;
        if (cost < best)
        {
            best = cost;
            pick = sh.id;
        }
    }
    // Grouped: m_expected rows in a group on average (g.M is their bound); up to three 128-row tiles the groups' last ones decide.  32 groups of 8096 rows: 128 x 256 151 us against 160 for
    // 128 x 128 and 167 for 256 x 192 (N 2816, K 2048); of 1944 rows 128 x 128 92 us, the wider ones 95 and more.  256 x 256 only where it saves rounds; a round of the last few tiles,
    // most of them nearly empty, does not count against the smaller ones.
    if (m_expected > 0 && m_expected <= 384)
    {
        auto cost = [&](int bm, double f, double rest) { return std::ceil(expected_tiles(m_expected, bm) * g.batch * ((g.N + 255) / 256) / cus - rest) * bm * f; };
        pick = m_expected <= 64 ? 0 : cost(256, shapes[2].f, 0.02) < cost(128, shapes[3].f, 0.08) ? 2 : 3;
    }
    // Up to two tall tiles of rows of 512 values and more, where K-tiles count and not a tile's start (and which the times are fitted to): by time.  Of more than 384 rows the shapes
    // above, too (16 groups of 453, 512, 1024 128 x 128 15.2 us, 128 x 256 20.7).
    if (served && m_expected > 0 && m_expected <= 2 * wide::TALL_BM && g.K >= 512)
    {
        const GroupForm form = pick_group_form(g, m_expected);
        if (form == GROUP_TALL)
            return wide::launch_tall(g, stream);
        if (form == GROUP_256x256)
            return wide::launch<W_BF16>(g, stream);
        if (m_expected <= 384)
            pick = form == GROUP_128x128 ? 0 : 3;
    }
    // 256 x 256 tiles of gemm_wide_impl.h
    if (served)
    {
        if (m_expected > 0)
        {
            // rounds of all groups' tiles, the last one of a group being there as often as not
            auto tiles = [&](int bm, int bn) { return (std::ceil(m_expected / (double) bm) + 0.4) * g.batch * ((g.N + bn - 1) / bn) / cus; };
            const Shape& sh = shapes[pick];
            const double kt = g.K / 64;
            if (m_expected >= 384 && std::max(1.0, tiles(256, 256)) * (kt * 0.85 + 1.5) + 4.0 < std::max(1.0, tiles(sh.bm, sh.bn)) * (kt * sh.bm * sh.bn * sh.f / 65536.0 + 4.0))
                return wide::launch<W_BF16>(g, stream);
        }
        else if (!g.group_off)
        {
            const Shape& sh = shapes[pick];
            const int64_t tiles = (int64_t) ((g.M + sh.bm - 1) / sh.bm) * ((g.N + sh.bn - 1) / sh.bn) * (g.batch > 1 ? g.batch : 1);
            // (a round of the lock-step tiles pays its first requests and its results each time: 2.5 K-tiles)
            if (wide::cost(g, 2) < (double) ((tiles + cus - 1) / cus) * ((double) (g.K / 64) * sh.bm * sh.bn * sh.f / 65536.0 + 2.5))
                return wide::launch<W_BF16>(g, stream);
        }
    }
    if (served)
        switch (pick)
        {
        case 0: return wide::launch_row128<2, 4, 2, 1, 4, false>(g, stream);
        case 3: return wide::launch_row128<2, 4, 2, 2, 3, true>(g, stream);
        case 4: return wide::launch_row128<4, 2, 1, 3, 4, true>(g, stream);
        case 5: return wide::launch_row128<4, 2, 1, 1, 4, false>(g, stream);
        }
    if (g.act == ACT_SCALE_CAP || g.act == ACT_GELU_MUL)
        pick = 0; // the shape whose epilogue has them
    const int gated = g.act >= ACT_GATE_SILU ? (g.seam.n_sec > 0 ? g.seam.sec[0].col0 : g.N) : 0;
    if ((gated & 15) || (gated && ((g.ldc & 7) || (reinterpret_cast<uintptr_t>(g.c) & 15) || g.out_dtype != DT_BFLOAT16)))
        pick = 0; // gated rows that do not leave in 16-byte pieces
    switch (pick)
    {
    case 1: return launch_cfg<W_BF16, 4, 2, 2, 3, 1, 128, 2>(g, stream);
    case 2: return launch_cfg<W_BF16, 2, 4, 4, 2, 1, 128, 2>(g, stream);
    case 3: return launch_cfg<W_BF16, 2, 4, 2, 2, 1, 128, 3>(g, stream);
    case 4: return launch_cfg<W_BF16, 4, 2, 1, 3, 1, 128, 4>(g, stream);
    case 5: return launch_cfg<W_BF16, 4, 2, 1, 1, 1, 128, 4>(g, stream);
    default: return launch_cfg<W_BF16, 2, 4, 2, 1, 1, 128, 4>(g, stream);
    }
}

} // namespace

bool stack_row_norm_serves(const StackRowNorm& n, int dtype, int width)
{
    auto pieces = [](const void* p) { return !(reinterpret_cast<uintptr_t>(p) & 15); };
    return dtype == DT_BF16 && width % 16 == 0 && width > 0 && width <= 4096 && (n.parts == 0 || ((n.parts == 1 || n.parts == 2 || n.parts == 4 || (n.parts == 8 && width % 2048 == 0)) && !n.y && !n.in)) && n.x && n.w && pieces(n.x) && pieces(n.y)
        && pieces(n.w) && pieces(n.w2) && pieces(n.h) && pieces(n.h2) && pieces(n.x_out) && (!n.y || (n.mix && n.out && n.x_out && n.x_out != n.x)) && (!n.h2 || (n.w2 && n.parts));
}

int launch_stack_row_gemm(const StackGemmParams& p_in, const StackRowNorm& n, hipStream_t stream)
{
    StackGemmParams p = p_in;
    if (p.ldw == 0)
        p.ldw = p.K;
    if (p.M != 1 || p.batch != 1 || p.group_off || p.a_rows || p.N <= 0 || !p.w || (!p.c && !p.resid) || !stack_row_norm_serves(n, p.dtype, p.K) || (reinterpret_cast<uintptr_t>(p.w) & 15)
        || p.ldw % 8 || p.ldw < p.K || p.ldw >= (1 << 26) || p.act == ACT_GELU_MUL || p.act == ACT_SCALE_CAP
        || (p.act >= ACT_GATE_SILU && (p.resid || ((p.seam.n_sec > 0 ? p.seam.sec[0].col0 : p.N) & 1))))
        return 1;
    const bool many = p.N > 16 * launch_util::device_cus(); // as in pick_row_shape
    auto go = [&](auto shape, auto np) {
        using S = decltype(shape);
        constexpr int NP = decltype(np)::value;
        auto in = [&](auto parts) { hipLaunchKernelGGL((row_norm_kernel<S::KS, S::NC, NP, decltype(parts)::value>), dim3((p.N + S::cols - 1) / S::cols), dim3(256), 0, stream, p, n); };
        switch (n.parts)
        {
        case 0: return in(std::integral_constant<int, 0>());
        case 1: return in(std::integral_constant<int, 1>());
        case 2: return in(std::integral_constant<int, 2>());
        case 4: return in(std::integral_constant<int, 4>());
        default:
            if constexpr (NP > 1)
                in(std::integral_constant<int, 8>());
        }
    };
    using Quarter1 = std::integral_constant<int, 1>; // pieces of a lane
    using Quarter2 = std::integral_constant<int, 2>;
    using Quarter4 = std::integral_constant<int, 4>;
    if (p.K <= 512)
        go(RowShape<1, 1>(), Quarter1());
    else if (p.K <= 1024)
        many ? go(RowShape<1, 2>(), Quarter1()) : go(RowShape<2, 1>(), Quarter1());
    else if (p.K <= 2048)
        many ? go(RowShape<1, 4>(), Quarter2()) : go(RowShape<4, 1>(), Quarter2());
    else
        p.N < 8 * launch_util::device_cus() ? go(RowShape<4, 2>(), Quarter4()) : go(RowShape<1, 8>(), Quarter4());
    return launched("stack_gemm row and norm");
}

bool stack_lone_serves(const StackMoeParams& m, const StackGemmParams& up, const StackGemmParams& down)
{
    auto rows_of_pieces = [](const StackGemmParams& p) {
        return p.K > 0 && p.N > 0 && p.K % 8 == 0 && p.lda % 8 == 0 && p.stride_w % 8 == 0 && p.ldw == 0 && p.c && !p.resid && !p.bias && p.seam.n_sec == 0
            && !((reinterpret_cast<uintptr_t>(p.a) | reinterpret_cast<uintptr_t>(p.w)) & 15) && (p.act < ACT_GATE_SILU || !(p.N & 1));
    };
    // (every wave of the first products makes all choices: with many of them that costs more than the launch it saves.  Steps of 3 layers of 64 experts, us,
    // in brackets with the ordering launch; width x ff 1024 x 704, 4 choices 161 - 164 (165 - 184), 8 172 - 175 (179 - 199), 16 214 - 216 (209 - 219), 64 776
    // (376); 2048 x 1408 172 - 186 (188 - 210), 230 - 233 (229 - 246), 312 - 315 (299 - 320), 1490 (740))
    return m.tokens == 1 && m.dtype == DT_BF16 && m.experts + m.identity <= LONE_OUT && m.top <= 8 && rows_of_pieces(up) && rows_of_pieces(down);
}

int launch_stack_lone_up(const StackMoeParams& m, const StackGemmParams& p_in, hipStream_t stream)
{
    StackGemmParams p = p_in;
    p.M = 1;
    p.ldw = p.K;
    pick_row_shape(p.N, p.K, m.top, true, [&](auto shape) {
        using S = decltype(shape);
        hipLaunchKernelGGL((lone_up_kernel<S::KS, S::NC>), dim3((p.N + S::cols - 1) / S::cols, 1, m.top), dim3(256), 0, stream, p, m);
    });
    return launched("stack_lone_up");
}

int launch_stack_lone_down(const StackMoeParams& m, const StackGemmParams& p_in, hipStream_t stream)
{
    StackGemmParams p = p_in;
    p.M = 1;
    p.ldw = p.K;
    pick_row_shape(p.N, p.K, m.top, true, [&](auto shape) {
        using S = decltype(shape);
        hipLaunchKernelGGL((lone_down_kernel<S::KS, S::NC>), dim3((p.N + S::cols - 1) / S::cols, 1, m.top), dim3(256), 0, stream, p, m.topk_idx, m.experts);
    });
    return launched("stack_lone_down");
}

int launch_stack_gemm(const StackGemmParams& p_in, hipStream_t stream)
{
    StackGemmParams p = p_in;
    if (p.M <= 0 || p.N <= 0)
        return 0;
    if (p.ldw == 0)
        p.ldw = p.K;
    if (p.K <= 0 || !p.a || !p.w || (!p.c && !p.resid))
    {
        set_error("stack_gemm: M %d N %d K %d with a missing operand", p.M, p.N, p.K);
        return -1;
    }
    if (p.dtype != DT_BF16 && p.dtype != DT_FLOAT)
    {
        set_error("stack_gemm: element type %d is not served (bfloat16 or float32)", p.dtype);
        return -1;
    }
    if (p.batch < 1 || (p.batch > 1 && p.resid) || (p.group_off && (p.resid || p.stride_a || p.stride_c))
        || (p.a_rows && !p.group_off) || (p.group_off && p.group_total < 1) || p.ldw < p.K || p.seam.n_sec < 0 || p.seam.n_sec > 2 || (p.seam.n_sec > 0 && (p.batch > 1 || p.group_off || p.resid))
        || (p.act == ACT_GELU_MUL && (!p.seam.mul || !p.seam.mul_rows || p.group_off))
        || (p.act >= ACT_GATE_SILU && (p.resid || p.split_ws || ((p.seam.n_sec > 0 ? p.seam.sec[0].col0 : p.N) & 1))))
    {
        set_error("stack_gemm: batch %d, act %d (a batched product has no residual seam and no output sections; a grouped one takes its rows from one a and one c)", p.batch, p.act);
        return -1;
    }
    const dim3 tiles((p.N + TN - 1) / TN, (p.M + TM - 1) / TM, p.batch);
    if (p.dtype == DT_FLOAT)
    {
        hipLaunchKernelGGL((fma_tile_kernel<DT_FLOAT>), tiles, dim3(256), 0, stream, p);
        return launched("stack_gemm fp32");
    }
    const bool aligned = !(reinterpret_cast<uintptr_t>(p.a) & 15) && !(reinterpret_cast<uintptr_t>(p.w) & 15) && p.K % 8 == 0 && p.lda % 8 == 0 && p.ldw % 8 == 0
        && (p.batch == 1 || (p.stride_a % 8 == 0 && p.stride_w % 8 == 0));
    if (aligned && p.M < 32 && p.ldw < (1 << 26))
    {
        const int cus = launch_util::device_cus();
        // a grouped step of few rows: as many products as groups can have rows
        const bool few = p.group_off && p.group_total < p.batch;
        const int products = few ? p.group_total : p.batch, groups = few ? p.batch : 0;
        if (p.M <= 1)
        {
            launch_row(p, products, groups, stream);
            return launched("stack_gemm row");
        }
        if (p.batch == 1 && !p.group_off && p.M <= 8 && (p.N + 7) / 8 * 2 <= cus && p.K >= 2048)
        {
            // us at 2 / 4 / 8 rows, in brackets slim_kernel: 256 x 2048 3.5 / 3.6 / 4.5 (4.8 / 4.8 / 4.9), 1024 x 2048 3.9 / 4.1 / 5.1 (5.0 / 5.0 / 5.1),
            // 1024 x 4096 5.0 / 5.3 / 6.7 (6.3 / 6.3 / 6.5)
            const dim3 kg((p.N + SK_R - 1) / SK_R);
            if (p.M <= 4)
                hipLaunchKernelGGL((skinny_ksplit_kernel<4>), kg, dim3(256), 0, stream, p);
            else
                hipLaunchKernelGGL((skinny_ksplit_kernel<8>), kg, dim3(256), 0, stream, p);
            return launched("stack_gemm skinny (K over waves)");
        }
        launch_slim(p, products, groups, stream);
        return launched("stack_gemm slim");
    }
    if (aligned && p.M >= 32 && p.batch == 1 && !p.group_off && p.K % 64 && p.K > 64 && (p.resid || (p.out_f32 && p.act == ACT_NONE && p.seam.n_sec == 0)))
    {
        // rows that end inside a 128-byte stage: the LDS-DMA tiles take the whole stages, plain FMAs add what is left of K (8 .. 56 columns, exact products,
        // bound by the fp32 result's way there and back) to it.  From one whole stage on quicker than the register-staged tiles, whose 64-byte slabs take
        // 2 us each whatever the shape, us at M x N x K, in brackets those: 292 x 1536 x 4128 34 (278), x 1376 21 (107), x 288 15 (39), x 72 12 (28);
        // 41 x 512 x 4128 31 (266); 4096 x 512 x 1376 30 (111); 4096 x 1536 x 4128 86 (755), x 72 32 (49).  16-bit results, which would be rounded
        // twice, stay with them.
        StackGemmParams whole = p, rest = p;
        whole.K = p.K / 64 * 64;
        rest.K = p.K - whole.K;
        rest.a = reinterpret_cast<const uint16_t*>(p.a) + whole.K;
        rest.w = reinterpret_cast<const uint16_t*>(p.w) + whole.K;
        rest.split_ws = nullptr;
        if (!p.resid)
        {
            rest.resid = reinterpret_cast<float*>(p.c);
            rest.ldr = p.ldc;
            rest.gate = nullptr;
        }
        if (launch_stack_gemm(whole, stream))
            return -1;
        hipLaunchKernelGGL((fma_tile_kernel<DT_BF16>), tiles, dim3(256), 0, stream, rest);
        return launched("stack_gemm rest of K");
    }
    const int64_t tiles128 = (int64_t) ((p.M + 127) / 128) * ((p.N + 127) / 128);
    if (aligned && p.split_ws && p.batch == 1 && p.M >= 32 && tiles128 * 2 <= launch_util::device_cus())
    {
        // few tiles: parts of K (whole 128-byte stages, at least 4 of them) until the chip is full
        int parts = 1;
        while (parts < 16 && tiles128 * parts * 2 <= launch_util::device_cus() && p.K % (64 * parts * 2) == 0 && p.K / (parts * 2) >= 256
            && (int64_t) parts * 2 * p.M * p.N <= p.split_floats)
            parts *= 2;
        if (parts > 1)
        {
            StackGemmParams part;
            part.dtype = p.dtype;
            part.out_f32 = 1;
            part.M = p.M;
            part.N = p.N;
            part.K = p.K / parts;
            part.a = p.a;
            part.lda = p.lda;
            part.w = p.w;
            part.ldw = p.ldw;
            part.c = p.split_ws;
            part.ldc = p.N;
            part.batch = parts;
            part.stride_a = part.stride_w = part.K;
            part.stride_c = (int64_t) p.M * p.N;
            if (launch_stack_gemm(part, stream))
                return -1;
            hipLaunchKernelGGL(split_sum_kernel, dim3((unsigned) (((int64_t) p.M * p.N + 255) / 256)), dim3(256), 0, stream, p, p.split_ws, parts);
            return launched("stack_gemm split sum");
        }
    }
    if (aligned && (!p.group_off || p.K % 64 == 0))
    {
        // the LDS-DMA tiles take a batch in one launch (blockIdx.y); the register-staged tiles one product per launch (and no
        // groups: their row count is the device's)
        const bool glds = (p.M >= 32 || p.group_off) && p.K % 64 == 0;
        const int launches = glds ? 1 : p.batch;
        int rc = 0;
        for (int b = 0; b < launches && rc == 0; ++b)
        {
            GemmParams g;
            g.wtype = W_BF16;
            g.out_dtype = p.out_f32 ? DT_FLOAT : DT_BFLOAT16;
            g.M = p.M;
            g.N = p.N;
            g.K = p.K;
            g.a = reinterpret_cast<const char*>(p.a) + (int64_t) b * p.stride_a * 2;
            g.lda = p.lda;
            g.w = reinterpret_cast<const char*>(p.w) + (int64_t) b * p.stride_w * 2;
            g.ldw = p.ldw * 2;
            g.c = p.c ? reinterpret_cast<char*>(p.c) + (int64_t) b * p.stride_c * (p.out_f32 ? 4 : 2) : nullptr;
            g.ldc = p.ldc;
            g.resid = p.resid;
            g.ldr = p.ldr;
            g.gate = p.gate;
            g.ldg = p.ldg;
            g.gate_bias = p.gate_bias;
            g.bias = p.bias;
            g.act = p.act;
            g.seam = p.seam;
            g.a_rows = p.a_rows;
            if (glds)
            {
                g.batch = p.batch;
                g.batch_a = p.stride_a * 2;
                g.batch_w = p.stride_w * 2;
                g.batch_c = p.stride_c * (p.out_f32 ? 4 : 2);
                g.group_off = p.group_off;
                g.group_total = p.group_total;
                rc = launch_glds_bf16(g, stream, p.group_off ? p.group_rows : 0);
            }
            else
                rc = launch_gemm_mfma(g, stream);
        }
        if (rc <= 0)
            return rc;
    }
    hipLaunchKernelGGL((fma_tile_kernel<DT_BF16>), tiles, dim3(256), 0, stream, p);
    return launched("stack_gemm bf16 fma tiles");
}

} // namespace kernels
} // namespace tllm
