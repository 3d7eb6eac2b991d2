// Routed mixture of experts of the ragged-batch stack engine (stack_kernels.h): the fp32 router with its grouped top-k choice,
// the ordering of (token, chosen expert) pairs by expert for the grouped products, and the weighted sum of the experts' outputs.
#include "dev_utils.h"
#include "launch_util.h"
#include "stack_kernels.h"
#include "stack_norm_impl.h"
#include "stack_route_impl.h"
#include <algorithm>

namespace tllm
{
namespace kernels
{
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
__device__ __forceinline__ void st_el(void* p, int64_t i, float v)
{
    if constexpr (DT == DT_BF16)
        reinterpret_cast<uint16_t*>(p)[i] = f2bf(v);
    else
        reinterpret_cast<float*>(p)[i] = v;
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

constexpr int RT = 8;         // tokens per logits workgroup: a router row is read once for all of them
constexpr int MAX_OUT = 1024; // router outputs (experts + identities)
constexpr int MAX_TOP = 64;
constexpr int RANKED_PAIRS = 64; // pairs up to which every thread compares all of them
constexpr int FEW_TOKENS = RT; // steps of this many tokens or fewer are routed and ordered in one launch (and gather inside it)

// acc[r] = this lane's share of router row e times the rows t0 .. t0 + nt of h; lanes split the width in float4 pieces where rows are
// 16-byte aligned
template <int DT, int NR = RT>
__device__ __forceinline__ void router_row(const StackMoeParams& p, int e, int t0, int nt, int lane, float (&acc)[NR])
{
    const int W = p.width;
#pragma unroll
    for (int r = 0; r < NR; ++r)
        acc[r] = 0.f;
    const float* wr = p.router_w + (int64_t) e * W;
    if ((W & 7) == 0)
    {
        // AHEAD pieces of the row are requested before the first is used (a piece behind the row: its first one again, unused)
        constexpr int AHEAD = 4;
        for (int k0 = lane * 8; k0 < W; k0 += AHEAD * 64 * 8)
        {
            float4 w[AHEAD][2];
#pragma unroll
            for (int a = 0; a < AHEAD; ++a)
            {
                const int k = k0 + a * 64 * 8 < W ? k0 + a * 64 * 8 : k0;
                w[a][0] = *reinterpret_cast<const float4*>(wr + k);
                w[a][1] = *reinterpret_cast<const float4*>(wr + k + 4);
            }
#pragma unroll
            for (int r = 0; r < NR; ++r)
            {
                if (r >= nt)
                    break;
                float hv[AHEAD][8];
#pragma unroll
                for (int a = 0; a < AHEAD; ++a)
                {
                    const int k = k0 + a * 64 * 8 < W ? k0 + a * 64 * 8 : k0;
                    if constexpr (DT == DT_BF16)
                    {
                        const uint4 u = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(p.h) + (int64_t) (t0 + r) * W + k);
                        const uint32_t us[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                        {
                            hv[a][2 * i] = __builtin_bit_cast(float, us[i] << 16);
                            hv[a][2 * i + 1] = __builtin_bit_cast(float, us[i] & 0xffff0000u);
                        }
                    }
                    else
                    {
                        const float* hp = reinterpret_cast<const float*>(p.h) + (int64_t) (t0 + r) * W + k;
                        const float4 h0 = *reinterpret_cast<const float4*>(hp), h1 = *reinterpret_cast<const float4*>(hp + 4);
                        hv[a][0] = h0.x, hv[a][1] = h0.y, hv[a][2] = h0.z, hv[a][3] = h0.w;
                        hv[a][4] = h1.x, hv[a][5] = h1.y, hv[a][6] = h1.z, hv[a][7] = h1.w;
                    }
                }
#pragma unroll
                for (int a = 0; a < AHEAD; ++a)
                {
                    if (k0 + a * 64 * 8 >= W)
                        break;
                    const float wv[8] = {w[a][0].x, w[a][0].y, w[a][0].z, w[a][0].w, w[a][1].x, w[a][1].y, w[a][1].z, w[a][1].w};
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        acc[r] = fmaf(wv[i], hv[a][i], acc[r]);
                }
            }
        }
    }
    else
    {
        for (int k = lane; k < W; k += 64)
        {
            const float wv = wr[k];
#pragma unroll
            for (int r = 0; r < NR; ++r)
                if (r < nt)
                    acc[r] = fmaf(wv, ld_el<DT>(p.h, (int64_t) (t0 + r) * W + k), acc[r]);
        }
    }
}

// Router logits, fp32: workgroup (x, y) = 4 router rows (one per wave) x NR tokens (one: a lone token's, without the
// code of eight, which such a launch spends its time fetching).  z [tokens, outputs].
template <int DT, int NR>
__global__ __launch_bounds__(256) void moe_logits_kernel(const StackMoeParams p, float* z)
{
    const int NE = p.experts + p.identity;
    const int e = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, t0 = blockIdx.y * NR;
    if (e >= NE)
        return;
    const int nt = NR > 1 && p.tokens - t0 < NR ? p.tokens - t0 : NR;
    float acc[NR];
    router_row<DT, NR>(p, e, t0, nt, lane, acc);
#pragma unroll
    for (int r = 0; r < NR; ++r)
    {
        const float sum = wave_sum(acc[r]);
        if (lane == 0 && r < nt)
            z[(int64_t) (t0 + r) * NE + e] = sum;
    }
}

// A lone token's, its row formed here (StackRowNorm) while the router's rows are under way: lane l has values 8 l .. of every 512, in the order of router_row.
// 34 outputs of width 2048 in a step: 3.5 us for what took 2.3 and 3.3.
template <int NP>
__global__ __launch_bounds__(256) void moe_logits_norm_kernel(const StackMoeParams p, const StackRowNorm n)
{
    constexpr int PIECES = 2 * NP; // of 512 values, all requested at once
    __shared__ __attribute__((aligned(16))) uint16_t row[NP * 1024];
    __shared__ __attribute__((aligned(16))) float red[LoneRow<NP, 0>::SUMS];
    const int NE = p.experts + p.identity, W = p.width, lane = threadIdx.x & 63, e = blockIdx.x * 4 + (threadIdx.x >> 6);
    LoneRow<NP, 0> lone;
    lone.request(n, W);
    const float* wr = p.router_w + (int64_t) (e < NE ? e : NE - 1) * W;
    float4 w[PIECES][2];
#pragma unroll
    for (int a = 0; a < PIECES; ++a)
    {
        const int k = a * 512 + lane * 8 < W ? a * 512 + lane * 8 : 0;
        w[a][0] = *reinterpret_cast<const float4*>(wr + k);
        w[a][1] = *reinterpret_cast<const float4*>(wr + k + 4);
    }
    lone.finish(n, W, row, red, blockIdx.x == 0);
    float acc = 0.f;
#pragma unroll
    for (int a = 0; a < PIECES; ++a)
    {
        const int k = a * 512 + lane * 8;
        const uint4 u = *reinterpret_cast<const uint4*>(row + (k < W ? k : 0));
        const uint32_t us[4] = {u.x, u.y, u.z, u.w};
        const float wv[8] = {w[a][0].x, w[a][0].y, w[a][0].z, w[a][0].w, w[a][1].x, w[a][1].y, w[a][1].z, w[a][1].w};
        if (k < W)
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                acc = fmaf(wv[2 * i], __builtin_bit_cast(float, us[i] << 16), acc);
                acc = fmaf(wv[2 * i + 1], __builtin_bit_cast(float, us[i] & 0xffff0000u), acc);
            }
    }
    acc = wave_sum(acc);
    if (lane == 0 && e < NE)
        p.logits[e] = acc;
}

// The same for prompts through fp32 matrix products: workgroup (x, y) = 16 tokens x 16 router rows, its 8 waves share the width, AHEAD
// pieces of 32 values requested at a time, and meet in LDS.  Lane (r, g) holds values 8 g .. 8 g + 7 of a piece of row r of both operands;
// product j of a piece takes value j of every lane, since the order of a sum's terms is free.  Bound by what a CU draws of both operands.  1672
// tokens, 32 outputs of width 2048 in a prompt: 27.5 us by dot products, 10.9 here.
template <int DT>
__global__ __launch_bounds__(512) void moe_logits_mfma_kernel(const StackMoeParams p, float* z)
{
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    constexpr int AHEAD = 4;
    __shared__ f32x4 part[8][64];
    const int NE = p.experts + p.identity, W = p.width, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int row = lane & 15, g = lane >> 4, t0 = blockIdx.y * 16, e = blockIdx.x * 16 + row;
    const int64_t arow = (int64_t) (t0 + row < p.tokens ? t0 + row : p.tokens - 1) * W + 8 * g;
    const float* wrow = p.router_w + (int64_t) (e < NE ? e : NE - 1) * W + 8 * g;
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k0 = wid * 32; k0 < W; k0 += AHEAD * 8 * 32)
    {
        uint4 a[AHEAD][DT == DT_BF16 ? 1 : 2];
        f32x4 b[AHEAD][2];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) // (a piece behind the row: the first one again, unused)
        {
            const int k = k0 + i * 8 * 32 < W ? k0 + i * 8 * 32 : k0;
            b[i][0] = *reinterpret_cast<const f32x4*>(wrow + k);
            b[i][1] = *reinterpret_cast<const f32x4*>(wrow + k + 4);
            if constexpr (DT == DT_BF16)
                a[i][0] = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(p.h) + arow + k);
            else
            {
                a[i][0] = *reinterpret_cast<const uint4*>(reinterpret_cast<const float*>(p.h) + arow + k);
                a[i][1] = *reinterpret_cast<const uint4*>(reinterpret_cast<const float*>(p.h) + arow + k + 4);
            }
        }
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
        {
            if (k0 + i * 8 * 32 >= W)
                break;
            float av[8];
            if constexpr (DT == DT_BF16)
            {
                const uint32_t us[4] = {a[i][0].x, a[i][0].y, a[i][0].z, a[i][0].w};
#pragma unroll
                for (int j = 0; j < 4; ++j)
                {
                    av[2 * j] = __builtin_bit_cast(float, us[j] << 16);
                    av[2 * j + 1] = __builtin_bit_cast(float, us[j] & 0xffff0000u);
                }
            }
            else
            {
                const uint32_t us[8] = {a[i][0].x, a[i][0].y, a[i][0].z, a[i][0].w, a[i][1].x, a[i][1].y, a[i][1].z, a[i][1].w};
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    av[j] = __builtin_bit_cast(float, us[j]);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av[j], b[i][j >> 2][j & 3], acc, 0, 0, 0);
        }
    }
    part[wid][lane] = acc;
    __syncthreads();
    if (wid != 0)
        return;
#pragma unroll
    for (int w = 1; w < 8; ++w)
        acc += part[w][lane];
    // lane (col, g) of the result holds rows 4 g .. 4 g + 3 of column col
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (e < NE && t0 + 4 * g + r < p.tokens)
            z[(int64_t) (t0 + 4 * g + r) * NE + e] = acc[r];
}

// One wave finishes one token: zr [outputs] holds its logits with the bias (LDS) and leaves as scores, cr [outputs] holds the corrections
// and leaves as choice values,
// lane k < top gets choice k.
__device__ __forceinline__ int select_token(const StackMoeParams& p, float* zr, float* cr, int lane, int t)
{
    const int NE = p.experts + p.identity;
    if (p.score == ROUTE_SIGMOID)
    {
        // every output's score by itself
        for (int e = lane; e < NE; e += 64)
        {
            const float s = 1.f / (1.f + expf(-zr[e]));
            zr[e] = s;
            cr[e] += s;
        }
    }
    else
    {
        float mx = -INFINITY;
        for (int e = lane; e < NE; e += 64)
            mx = fmaxf(mx, zr[e]);
        mx = wave_max(mx);
        float sum = 0.f;
        for (int e = lane; e < NE; e += 64)
        {
            const float x = expf(zr[e] - mx);
            zr[e] = x;
            sum += x;
        }
        sum = wave_sum(sum);
        const float inv = 1.f / sum;
        for (int e = lane; e < NE; e += 64)
        {
            const float s = zr[e] * inv;
            zr[e] = s;
            cr[e] += s;
        }
    }
    __builtin_amdgcn_wave_barrier();
    const int GC = p.group_count, GS = NE / GC;
    if (GC > 1 && p.group_keep < GC)
    {
        // a group's value: its largest choice value; the group_keep best groups stay, the others' experts cannot be chosen
        float gv[(MAX_OUT + 63) / 64];
        const int per_lane = (GC + 63) / 64;
        for (int i = 0; i < per_lane; ++i)
        {
            const int g = lane + i * 64;
            float m = -INFINITY;
            if (g < GC)
                for (int j = 0; j < GS; ++j)
                    m = fmaxf(m, cr[g * GS + j]);
            gv[i] = m;
        }
        bool kept[(MAX_OUT + 63) / 64];
        for (int i = 0; i < per_lane; ++i)
            kept[i] = false;
        for (int k = 0; k < p.group_keep; ++k)
        {
            float bv = -INFINITY;
            int bi = 0x7fffffff;
            for (int i = 0; i < per_lane; ++i)
            {
                const int g = lane + i * 64;
                if (g < GC && !kept[i] && (gv[i] > bv || (gv[i] == bv && g < bi)))
                {
                    bv = gv[i];
                    bi = g;
                }
            }
            wave_argmax(bv, bi);
            for (int i = 0; i < per_lane; ++i)
                if (lane + i * 64 == bi)
                    kept[i] = true;
        }
        for (int i = 0; i < per_lane; ++i)
        {
            const int g = lane + i * 64;
            if (g < GC && !kept[i])
                for (int j = 0; j < GS; ++j)
                    cr[g * GS + j] = -INFINITY;
        }
        __builtin_amdgcn_wave_barrier();
    }
    float mine = 0.f, total = 0.f; // lane k keeps choice k and its score; every lane the scores' sum
    int chosen = 0;
    for (int k = 0; k < p.top; ++k)
    {
        float bv = -INFINITY;
        int bi = 0x7fffffff;
        for (int e = lane; e < NE; e += 64)
        {
            const float c = cr[e];
            if (c > bv || (c == bv && e < bi && c > -INFINITY))
            {
                bv = c;
                bi = e;
            }
        }
        wave_argmax(bv, bi);
        if (bi >= NE) // fewer choosable experts than `top`: the place stays empty (weight 0 on an identity)
            bi = NE - 1, bv = -INFINITY;
        const float s = bv == -INFINITY ? 0.f : zr[bi];
        total += s;
        if (lane == k)
        {
            mine = s;
            chosen = bi;
        }
        if (lane == 0)
            cr[bi] = -INFINITY;
        __builtin_amdgcn_wave_barrier();
    }
    if (lane < p.top)
        p.topk_w[(int64_t) t * p.top + lane] = (p.normalize ? mine / (total + 1e-20f) : mine) * p.scale;
    return chosen;
}

// One wave per token (4 per workgroup): softmax over the logits, choice values, the kept groups, the top-k among them.
__global__ __launch_bounds__(256) void moe_select_kernel(const StackMoeParams p, const float* zg)
{
    extern __shared__ float sm[];
    const int NE = p.experts + p.identity;
    float* z = sm;              // [4][NE] scores
    float* ch = z + 4 * NE;     // [4][NE] choice values
    const int t0 = blockIdx.x * 4, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (t0 + wid < p.tokens)
        for (int e = lane; e < NE; e += 64)
        {
            z[wid * NE + e] = zg[(int64_t) (t0 + wid) * NE + e] + (p.bias ? p.bias[e] : 0.f);
            ch[wid * NE + e] = p.correction ? p.correction[e] : 0.f;
        }
    __syncthreads();
    const int t = t0 + wid;
    if (t >= p.tokens)
        return;
    const int chosen = select_token(p, z + wid * NE, ch + wid * NE, lane, t);
    if (lane < p.top)
        p.topk_idx[(int64_t) t * p.top + lane] = chosen;
}

// dst[:] = w * src[:] over one row of the element type (the weight of a pair applied to the expert's input), thread `i` of `n`
__device__ __forceinline__ void scaled_row(const StackMoeParams& p, char* dst, const char* src, float w, int i, int n)
{
    if (p.dtype == DT_BF16 && (p.width & 7) == 0) // (16-byte rows of 16-byte operands: h and a_sorted are allocations)
        for (int c = i * 8; c < p.width; c += n * 8)
        {
            const uint4 u = *reinterpret_cast<const uint4*>(src + c * 2);
            const uint32_t us[4] = {u.x, u.y, u.z, u.w};
            uint32_t o[4];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                o[k] = (uint32_t) f2bf(w * __builtin_bit_cast(float, us[k] << 16))
                    | ((uint32_t) f2bf(w * __builtin_bit_cast(float, us[k] & 0xffff0000u)) << 16);
            *reinterpret_cast<uint4*>(dst + c * 2) = make_uint4(o[0], o[1], o[2], o[3]);
        }
    else if (p.dtype == DT_BF16)
        for (int c = i; c < p.width; c += n)
            reinterpret_cast<uint16_t*>(dst)[c] = f2bf(w * bf2f(reinterpret_cast<const uint16_t*>(src)[c]));
    else
        for (int c = i; c < p.width; c += n)
            reinterpret_cast<float*>(dst)[c] = w * reinterpret_cast<const float*>(src)[c];
}

// The rows of few pairs are copied by the launch that orders them, a wave per pair, instead of by one of their own
__device__ __forceinline__ void gather_pairs(const StackMoeParams& p, int gather_row_bytes)
{
    const int pairs = p.tokens * p.top, NT = blockDim.x, lane = threadIdx.x & 63;
    for (int i = threadIdx.x >> 6; i < pairs; i += NT >> 6)
    {
        const int slot = p.slot_of_pair[i];
        if (slot < 0)
            continue;
        const char* src = reinterpret_cast<const char*>(p.h) + (int64_t) (i / p.top) * gather_row_bytes;
        char* dst = reinterpret_cast<char*>(p.a_sorted) + (int64_t) slot * gather_row_bytes;
        if (p.weight_input)
            scaled_row(p, dst, src, p.topk_w[i], lane, 64);
        else if ((gather_row_bytes & 15) == 0)
            for (int b = lane * 16; b < gather_row_bytes; b += 64 * 16)
                *reinterpret_cast<uint4*>(dst + b) = *reinterpret_cast<const uint4*>(src + b);
        else
            for (int b = lane * 2; b < gather_row_bytes; b += 64 * 2)
                *reinterpret_cast<uint16_t*>(dst + b) = *reinterpret_cast<const uint16_t*>(src + b);
    }
}

// One workgroup: counts per expert, offsets, a slot per pair.  Which of an expert's slots a pair gets depends on the order of the
// atomics; a row's product does not depend on its neighbours in a tile, so the results do not.  choice [tokens * top]: the chosen
// outputs; si: LDS, 2 * experts + 1 ints.
__device__ __forceinline__ void sort_pairs(const StackMoeParams& p, const int* choice, int gather_row_bytes, int* si)
{
    int* cnt = si;                  // [experts]
    int* off = cnt + p.experts;     // [experts + 1]
    const int pairs = p.tokens * p.top, tid = threadIdx.x, NT = blockDim.x;
    for (int e = tid; e < p.experts; e += NT)
        cnt[e] = 0;
    __syncthreads();
    for (int i = tid; i < pairs; i += NT)
    {
        const int e = choice[i];
        if (e < p.experts)
            atomicAdd(&cnt[e], 1);
    }
    __syncthreads();
    if (tid < 64) // one wave sums the counts, 64 experts at a time
    {
        int run = 0;
        for (int e0 = 0; e0 < p.experts; e0 += 64)
        {
            const int e = e0 + tid, own = e < p.experts ? cnt[e] : 0;
            int upto = own;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1)
            {
                const int below = __shfl_up(upto, d, 64);
                upto += tid >= d ? below : 0;
            }
            if (e < p.experts)
                off[e] = run + upto - own;
            run += __builtin_amdgcn_readlane(upto, 63);
        }
        if (tid == 0)
            off[p.experts] = run;
    }
    __syncthreads();
    for (int e = tid; e <= p.experts; e += NT)
    {
        p.group_off[e] = off[e];
        if (e < p.experts)
            cnt[e] = 0;
    }
    const int used = off[p.experts];
    for (int i = used + tid; i < pairs; i += NT)
        p.pair_of_slot[i] = -1;
    __syncthreads();
    for (int i = tid; i < pairs; i += NT)
    {
        const int e = choice[i];
        int slot = -1;
        if (e < p.experts)
        {
            slot = off[e] + atomicAdd(&cnt[e], 1);
            p.pair_of_slot[slot] = i;
            if (p.tok_of_slot)
                p.tok_of_slot[slot] = i / p.top;
        }
        p.slot_of_pair[i] = slot;
    }
    if (gather_row_bytes <= 0)
        return;
    __syncthreads();
    gather_pairs(p, gather_row_bytes);
}

// The same for a few pairs: an expert's first slot is how many pairs chose a lower one, a pair's slot counts the equal ones ahead of it.
// Every thread reads all choices, which no barrier or atomic separates: they cost less than the counting form's five barriers.
__device__ __forceinline__ void rank_pairs(const StackMoeParams& p, const int* choice, int gather_row_bytes)
{
    const int pairs = p.tokens * p.top, tid = threadIdx.x, NT = blockDim.x;
    for (int e = tid; e <= p.experts; e += NT)
    {
        int below = 0;
        for (int j = 0; j < pairs; ++j)
            below += choice[j] < e ? 1 : 0;
        p.group_off[e] = below;
    }
    for (int i = tid; i < pairs; i += NT)
    {
        const int own = choice[i];
        int below = 0, used = 0;
        for (int j = 0; j < pairs; ++j)
        {
            const int c = choice[j];
            below += (c < own || (c == own && j < i)) ? 1 : 0;
            used += c < p.experts ? 1 : 0;
        }
        const bool routed = own < p.experts;
        p.slot_of_pair[i] = routed ? below : -1;
        if (routed)
        {
            p.pair_of_slot[below] = i;
            if (p.tok_of_slot)
                p.tok_of_slot[below] = i / p.top;
        }
        if (i >= used)
            p.pair_of_slot[i] = -1;
    }
    if (gather_row_bytes <= 0)
        return;
    __syncthreads();
    gather_pairs(p, gather_row_bytes);
}

__global__ __launch_bounds__(1024) void moe_sort_kernel(const StackMoeParams p, int gather_row_bytes)
{
    extern __shared__ int si[];
    sort_pairs(p, p.topk_idx, gather_row_bytes, si);
}

// LDS of a launch that chooses for a few tokens and orders their pairs: scores and choice values first, then counts and choices
inline size_t plan_lds_bytes(const StackMoeParams& p)
{
    const size_t NE = (size_t) (p.experts + p.identity), T = (size_t) p.tokens;
    return sizeof(int) * std::max(2 * NE * T, 2 * (size_t) p.experts + 1 + T * (size_t) p.top);
}

// Wave t finishes token t, then the workgroup orders the pairs.  SPREAD: the logits come from other workgroups of this launch, bias and
// corrections are in LDS already.
template <bool SPREAD>
__device__ __forceinline__ void plan_few(const StackMoeParams& p, int gather_row_bytes, float* sm)
{
    const int NE = p.experts + p.identity, lane = threadIdx.x & 63, t = threadIdx.x >> 6;
    int* choice = reinterpret_cast<int*>(sm) + 2 * p.experts + 1;
    int chosen = 0;
    if (t < p.tokens)
    {
        float* z = sm + (int64_t) t * 2 * NE;
        for (int e = lane; e < NE; e += 64)
        {
            const float* src = p.logits + (int64_t) t * NE + e;
            if constexpr (SPREAD)
                z[e] += __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            else
            {
                z[e] = *src + (p.bias ? p.bias[e] : 0.f);
                z[NE + e] = p.correction ? p.correction[e] : 0.f;
            }
        }
        __builtin_amdgcn_wave_barrier();
        chosen = select_token(p, z, z + NE, lane, t);
    }
    __syncthreads(); // the scores' place is free
    if (t < p.tokens && lane < p.top)
        choice[t * p.top + lane] = chosen;
    __syncthreads();
    if (p.tokens * p.top <= RANKED_PAIRS)
        rank_pairs(p, choice, gather_row_bytes);
    else
        sort_pairs(p, choice, gather_row_bytes, reinterpret_cast<int*>(sm));
}

// Few tokens whose logits are there already.
__global__ __launch_bounds__(1024) void moe_plan_few_kernel(const StackMoeParams p, int gather_row_bytes)
{
    extern __shared__ float sm[];
    plan_few<false>(p, gather_row_bytes, sm);
}

// The same with the logits computed here, a router row per wave.  The rows are spread over workgroups, and the last one to arrive chooses
// and orders: a logit is written through to where every XCD sees it and waited for before its workgroup takes a ticket, the last one
// reads them past its own caches, and the ticket word is zero again for the next launch.  Bound by latencies in a row (row, ticket,
// logits, choices).  One workgroup for all rows draws too little bandwidth: one token, top 4, us alone / spread: 32 outputs of width
// 1024 8.2 / 7.6, 64 of 2048 13.7 / 8.1, 256 of 4096 110 / 13.5; eight tokens 15.6 / 12.8, 38 / 15.4, 295 / 25.  In a decode step
// (cold rows), 40 outputs of width 2048: 14.7 as a one-workgroup router and a sort, 9.8 here.
template <int DT>
__global__ __launch_bounds__(512) void moe_route_few_kernel(const StackMoeParams p, int gather_row_bytes)
{
    extern __shared__ float sm[];
    __shared__ uint32_t ticket;
    const int NE = p.experts + p.identity, lane = threadIdx.x & 63, e = blockIdx.x * 8 + (threadIdx.x >> 6);
    // what the choice adds to the logits comes in under the product
    for (int i = threadIdx.x; i < NE; i += 512)
    {
        const float b = p.bias ? p.bias[i] : 0.f, c = p.correction ? p.correction[i] : 0.f;
        for (int t = 0; t < p.tokens; ++t)
        {
            sm[t * 2 * NE + i] = b;
            sm[t * 2 * NE + NE + i] = c;
        }
    }
    if (e < NE)
    {
        float acc[RT];
        router_row<DT>(p, e, 0, p.tokens, lane, acc);
#pragma unroll
        for (int r = 0; r < RT; ++r)
            if (r < p.tokens)
            {
                const float sum = wave_sum(acc[r]);
                if (lane == 0)
                    __hip_atomic_store(p.logits + (int64_t) r * NE + e, sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0)
        ticket = __hip_atomic_fetch_add(p.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (ticket != gridDim.x - 1)
        return;
    if (threadIdx.x == 0)
        __hip_atomic_store(p.ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    plan_few<true>(p, gather_row_bytes, sm);
}

// a_sorted[slot, :] = h[token of the slot's pair, :]; 16 bytes per thread where the rows allow it
__global__ __launch_bounds__(256) void moe_gather_kernel(const StackMoeParams p, int row_bytes)
{
    const int slot = blockIdx.x;
    const int pair = p.pair_of_slot[slot];
    if (pair < 0)
        return;
    const char* src = reinterpret_cast<const char*>(p.h) + (int64_t) (pair / p.top) * row_bytes;
    char* dst = reinterpret_cast<char*>(p.a_sorted) + (int64_t) slot * row_bytes;
    if (p.weight_input)
        scaled_row(p, dst, src, p.topk_w[pair], threadIdx.x, 256);
    else if ((row_bytes & 15) == 0)
    {
        for (int i = threadIdx.x * 16; i < row_bytes; i += 256 * 16)
            *reinterpret_cast<uint4*>(dst + i) = *reinterpret_cast<const uint4*>(src + i);
    }
    else
    {
        for (int i = threadIdx.x * 2; i < row_bytes; i += 256 * 2)
            *reinterpret_cast<uint16_t*>(dst + i) = *reinterpret_cast<const uint16_t*>(src + i);
    }
}

// what scales the row that the experts' sum is added to
__device__ __forceinline__ float kept_share(const StackMoeParams& p, int t)
{
    return p.accumulate_gate ? 1.f / (1.f + expf(-p.accumulate_gate[t])) : 1.f;
}

template <int DT>
__global__ __launch_bounds__(256) void moe_combine_kernel(const StackMoeParams p, const float* ys, float* y)
{
    __shared__ int slot_s[MAX_TOP];
    __shared__ float w_s[MAX_TOP];
    const int t = blockIdx.x;
    if ((int) threadIdx.x < p.top)
    {
        slot_s[threadIdx.x] = p.slot_of_pair[(int64_t) t * p.top + threadIdx.x];
        w_s[threadIdx.x] = p.topk_w[(int64_t) t * p.top + threadIdx.x];
    }
    __syncthreads();
    const float keep = kept_share(p, t);
    for (int c = threadIdx.x; c < p.width; c += 256)
    {
        float acc = p.accumulate ? keep * y[(int64_t) t * p.width + c] : 0.f;
        for (int k = 0; k < p.top; ++k)
        {
            const int slot = slot_s[k];
            const float v = slot >= 0 ? ys[(int64_t) slot * p.width + c] : ld_el<DT>(p.h, (int64_t) t * p.width + c);
            acc = fmaf((p.weight_input && slot >= 0) ? 1.f : w_s[k], v, acc); // an input-weighted expert's output is summed as it is

        }
        y[(int64_t) t * p.width + c] = acc;
        if (p.y_el)
            st_el<DT>(p.y_el, (int64_t) t * p.width + c, acc);
    }
}

// The same for rows of whole 16-byte pieces: four channels per thread, the row's channels over workgroups (blockIdx.y), every expert's
// piece requested before the first is added.
template <int DT, int TOP>
__global__ __launch_bounds__(256) void moe_combine_vec_kernel(const StackMoeParams p, const float* ys, float* y)
{
    const int t = blockIdx.x, c = (blockIdx.y * 256 + threadIdx.x) * 4;
    if (c >= p.width)
        return;
    float4 acc = p.accumulate ? *reinterpret_cast<const float4*>(y + (int64_t) t * p.width + c) : make_float4(0.f, 0.f, 0.f, 0.f);
    if (p.accumulate_gate)
    {
        const float keep = kept_share(p, t);
        acc = make_float4(acc.x * keep, acc.y * keep, acc.z * keep, acc.w * keep);
    }
    for (int k0 = 0; k0 < p.top; k0 += TOP)
    {
        float4 v[TOP];
        float w[TOP];
#pragma unroll
        for (int k = 0; k < TOP; ++k)
        {
            const bool on = k0 + k < p.top;
            const int64_t pair = (int64_t) t * p.top + (on ? k0 + k : k0);
            const int slot = p.slot_of_pair[pair];
            w[k] = on ? ((p.weight_input && slot >= 0) ? 1.f : p.topk_w[pair]) : 0.f;
            if (slot >= 0)
                v[k] = *reinterpret_cast<const float4*>(ys + (int64_t) slot * p.width + c);
            else
            {
                const int64_t o = (int64_t) t * p.width + c;
                v[k] = make_float4(ld_el<DT>(p.h, o), ld_el<DT>(p.h, o + 1), ld_el<DT>(p.h, o + 2), ld_el<DT>(p.h, o + 3));
            }
        }
#pragma unroll
        for (int k = 0; k < TOP; ++k)
        {
            if (k0 + k >= p.top)
                break;
            acc.x = fmaf(w[k], v[k].x, acc.x);
            acc.y = fmaf(w[k], v[k].y, acc.y);
            acc.z = fmaf(w[k], v[k].z, acc.z);
            acc.w = fmaf(w[k], v[k].w, acc.w);
        }
    }
    const int64_t o = (int64_t) t * p.width + c;
    *reinterpret_cast<float4*>(y + o) = acc;
    if (p.y_el)
    {
        if constexpr (DT == DT_BF16)
            *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(p.y_el) + o)
                = make_uint2((uint32_t) f2bf(acc.x) | ((uint32_t) f2bf(acc.y) << 16), (uint32_t) f2bf(acc.z) | ((uint32_t) f2bf(acc.w) << 16));
        else
            *reinterpret_cast<float4*>(reinterpret_cast<float*>(p.y_el) + o) = acc;
    }
}

bool moe_ok(const StackMoeParams& p, const char* what)
{
    if (p.dtype != DT_BF16 && p.dtype != DT_FLOAT)
    {
        set_error("%s: element type %d is not served (bfloat16 or float32)", what, p.dtype);
        return false;
    }
    const int NE = p.experts + p.identity;
    if (p.experts < 1 || p.identity < 0 || NE > MAX_OUT || p.top < 1 || p.top > MAX_TOP || p.top > NE || p.group_count < 1 || NE % p.group_count
        || p.group_keep < 1 || p.group_keep > p.group_count || p.width < 1)
    {
        set_error("%s: %d experts + %d identities in %d groups of which %d are kept, top %d is not a router it serves (at most %d outputs, "
                  "top <= %d, equal groups)",
            what, p.experts, p.identity, p.group_count, p.group_keep, p.top, MAX_OUT, MAX_TOP);
        return false;
    }
    return true;
}

} // namespace

int launch_stack_moe_route(const StackMoeParams& p, hipStream_t stream)
{
    if (p.tokens <= 0)
        return 0;
    if (!moe_ok(p, "stack_moe_route"))
        return -1;
    if (!p.logits)
    {
        set_error("stack_moe_route: no room for the logits");
        return -1;
    }
    const int NE = p.experts + p.identity;
    if (p.have_logits)
    {
        hipLaunchKernelGGL(moe_select_kernel, dim3((p.tokens + 3) / 4), dim3(256), sizeof(float) * 2 * 4 * NE, stream, p, p.logits);
        return launched("stack_moe_select");
    }
    const dim3 lg((NE + 3) / 4, (p.tokens + RT - 1) / RT);
    // us with the choice behind it, dot products / matrix products: 256 tokens the same (32 outputs of width 1024 10.8 / 10.5, 64 of 4096
    // 19.6 / 19.8), 1672 tokens 15.9 / 10.7 and 73.5 / 28.5, 160 outputs of 4096 138.7 / 62.7
    if (p.width % 32 == 0 && p.tokens > 256 && !((reinterpret_cast<uintptr_t>(p.h) | reinterpret_cast<uintptr_t>(p.router_w)) & 15))
    {
        const dim3 mg((NE + 15) / 16, (p.tokens + 15) / 16);
        if (p.dtype == DT_BF16)
            hipLaunchKernelGGL((moe_logits_mfma_kernel<DT_BF16>), mg, dim3(512), 0, stream, p, p.logits);
        else
            hipLaunchKernelGGL((moe_logits_mfma_kernel<DT_FLOAT>), mg, dim3(512), 0, stream, p, p.logits);
    }
    else if (p.dtype == DT_BF16)
        hipLaunchKernelGGL((moe_logits_kernel<DT_BF16, RT>), lg, dim3(256), 0, stream, p, p.logits);
    else
        hipLaunchKernelGGL((moe_logits_kernel<DT_FLOAT, RT>), lg, dim3(256), 0, stream, p, p.logits);
    if (launched("stack_moe_logits"))
        return -1;
    hipLaunchKernelGGL(moe_select_kernel, dim3((p.tokens + 3) / 4), dim3(256), sizeof(float) * 2 * 4 * NE, stream, p, p.logits);
    return launched("stack_moe_select");
}

int launch_stack_moe_sort(const StackMoeParams& p, hipStream_t stream)
{
    if (p.tokens <= 0)
        return 0;
    if (!moe_ok(p, "stack_moe_sort"))
        return -1;
    if (p.weight_input && !p.a_sorted)
    {
        set_error("stack_moe_sort: input weights need room for the scaled rows");
        return -1;
    }
    const size_t lds = sizeof(int) * (2 * (size_t) p.experts + 1);
    const int row_bytes = p.a_sorted ? p.width * (p.dtype == DT_BF16 ? 2 : 4) : 0;
    const bool few = p.tokens <= FEW_TOKENS || !p.a_sorted;
    hipLaunchKernelGGL(moe_sort_kernel, dim3(1), dim3(1024), lds, stream, p, few ? row_bytes : 0);
    const int rc = launched("stack_moe_sort");
    if (rc || few)
        return rc;
    hipLaunchKernelGGL(moe_gather_kernel, dim3(p.tokens * p.top), dim3(256), 0, stream, p, row_bytes);
    return launched("stack_moe_gather");
}

int launch_stack_moe_logits(const StackMoeParams& p, hipStream_t stream)
{
    if (p.tokens <= 0)
        return 0;
    if (!moe_ok(p, "stack_moe_logits"))
        return -1;
    const dim3 lg((p.experts + p.identity + 3) / 4, p.tokens);
    if (p.dtype == DT_BF16)
        hipLaunchKernelGGL((moe_logits_kernel<DT_BF16, 1>), lg, dim3(256), 0, stream, p, p.logits);
    else
        hipLaunchKernelGGL((moe_logits_kernel<DT_FLOAT, 1>), lg, dim3(256), 0, stream, p, p.logits);
    return launched("stack_moe_logits");
}

int launch_stack_moe_logits(const StackMoeParams& p, const StackRowNorm& n, hipStream_t stream)
{
    if (p.tokens != 1 || n.parts || !stack_row_norm_serves(n, p.dtype, p.width) || !moe_ok(p, "stack_moe_logits"))
    {
        set_error("stack_moe_logits: %d tokens of width %d, or a missing operand", p.tokens, p.width);
        return -1;
    }
    const dim3 lg((p.experts + p.identity + 3) / 4);
    if (p.width <= 1024)
        hipLaunchKernelGGL((moe_logits_norm_kernel<1>), lg, dim3(256), 0, stream, p, n);
    else if (p.width <= 2048)
        hipLaunchKernelGGL((moe_logits_norm_kernel<2>), lg, dim3(256), 0, stream, p, n);
    else
        hipLaunchKernelGGL((moe_logits_norm_kernel<4>), lg, dim3(256), 0, stream, p, n);
    return launched("stack_moe_logits");
}

int launch_stack_moe_plan(const StackMoeParams& p, hipStream_t stream)
{
    if (p.tokens <= 0)
        return 0;
    if (p.tokens > FEW_TOKENS || !(p.have_logits || p.ticket))
        return (launch_stack_moe_route(p, stream) || launch_stack_moe_sort(p, stream)) ? -1 : 0;
    if (!moe_ok(p, "stack_moe_plan"))
        return -1;
    const size_t lds = plan_lds_bytes(p);
    if (!p.logits || (p.weight_input && !p.a_sorted) || lds > 64 * 1024)
    {
        set_error("stack_moe_plan: %d tokens x %d outputs, or a missing operand", p.tokens, p.experts + p.identity);
        return -1;
    }
    const int row_bytes = p.a_sorted ? p.width * (p.dtype == DT_BF16 ? 2 : 4) : 0;
    if (p.have_logits)
        hipLaunchKernelGGL(moe_plan_few_kernel, dim3(1), dim3(1024), lds, stream, p, row_bytes);
    else
    {
        const dim3 grid((p.experts + p.identity + 7) / 8);
        // (eight tokens of 1024 outputs take all of the default 64 KiB, and the kernel's ticket stands beside them)
        const void* fn = p.dtype == DT_BF16 ? reinterpret_cast<const void*>(&moe_route_few_kernel<DT_BF16>) : reinterpret_cast<const void*>(&moe_route_few_kernel<DT_FLOAT>);
        launch_util::ensure_dynamic_lds(fn, lds + sizeof(uint32_t));
        if (p.dtype == DT_BF16)
            hipLaunchKernelGGL((moe_route_few_kernel<DT_BF16>), grid, dim3(512), lds, stream, p, row_bytes);
        else
            hipLaunchKernelGGL((moe_route_few_kernel<DT_FLOAT>), grid, dim3(512), lds, stream, p, row_bytes);
    }
    return launched("stack_moe_plan");
}

int launch_stack_moe_combine(const StackMoeParams& p, const float* y_sorted, float* y, hipStream_t stream)
{
    if (p.tokens <= 0)
        return 0;
    if (!moe_ok(p, "stack_moe_combine"))
        return -1;
    const bool al16 = !((reinterpret_cast<uintptr_t>(y_sorted) | reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(p.y_el)) & 15);
    if (p.width % 4 == 0 && al16)
    {
        const dim3 grid(p.tokens, (p.width / 4 + 255) / 256);
        if (p.dtype == DT_BF16)
            hipLaunchKernelGGL((moe_combine_vec_kernel<DT_BF16, 4>), grid, dim3(256), 0, stream, p, y_sorted, y);
        else
            hipLaunchKernelGGL((moe_combine_vec_kernel<DT_FLOAT, 4>), grid, dim3(256), 0, stream, p, y_sorted, y);
        return launched("stack_moe_combine");
    }
    if (p.dtype == DT_BF16)
        hipLaunchKernelGGL((moe_combine_kernel<DT_BF16>), dim3(p.tokens), dim3(256), 0, stream, p, y_sorted, y);
    else
        hipLaunchKernelGGL((moe_combine_kernel<DT_FLOAT>), dim3(p.tokens), dim3(256), 0, stream, p, y_sorted, y);
    return launched("stack_moe_combine");
}

} // namespace kernels
} // namespace tllm
