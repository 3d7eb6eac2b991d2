// A lone token's normed row, formed by the workgroups that read it (stack_kernels.h, StackRowNorm): shared by its products (stack_gemm.hip) and its
// router's logits (stack_moe.hip).  Everything has internal linkage.
#pragma once
#include "dev_utils.h"
#include "stack_kernels.h"
#include <type_traits>

namespace tllm
{
namespace kernels
{
namespace
{
using namespace dev;

// x^2 + y^2 + z^2 + w^2 with its contraction written out, x^2 or y^2 rounded first: left to the compiler, which of the two turned over with the code around it, and with it the
// last bit of a norm.  A row's sum of squares has the same bits in every launch that forms it.
template <bool X_FIRST>
__device__ __forceinline__ float sum_squares4(const float4& v)
{
    const float xy = X_FIRST ? fmaf(v.y, v.y, v.x * v.x) : fmaf(v.x, v.x, v.y * v.y);
    return fmaf(v.w, v.w, fmaf(v.z, v.z, xy));
}

// the squares of a thread's values of a part, likewise: the second one's first
template <int N>
__device__ __forceinline__ float sum_squares(const float (&v)[N])
{
    float ss = v[0] * v[0];
    if constexpr (N > 1)
        ss = fmaf(v[0], v[0], v[1] * v[1]);
#pragma unroll
    for (int k = 2; k < N; ++k)
        ss = fmaf(v[k], v[k], ss);
    return ss;
}

// Both forms: request() asks for the row, ahead of the operands that it is to arrive before and without a branch that a load would wait behind; finish() leaves it in `row`, LDS
// [width] in bfloat16.  red: LDS, SUMS floats on 16 bytes.  first: this workgroup also leaves what later launches read.  The sums of squares run in the order of the launch whose place
// is taken, so that a row has the same bits either way; what that costs (a sum over a wave a piece instead of one in all) passes while the weights are under way.

// A row of one stream, as hyper_norm_vec_kernel: a lane's float4, 64 lanes, the 256 values of each wave in turn.  The workgroup's 4 waves have NP such pieces each.
template <int NP>
struct StreamRow
{
    static constexpr int SUMS = 4 * NP;
    float4 x[NP], y[NP], w[NP];
    float cm, co, ci;

    __device__ __forceinline__ static int piece(int width, int k, bool& on)
    {
        const int c = threadIdx.x + 256 * k;
        on = c < width >> 2;
        return on ? c : 0;
    }
    __device__ __forceinline__ void request(const StackRowNorm& n, int width)
    {
        const float* y_or_x = n.y ? n.y : n.x;
        cm = n.y ? n.mix[0] : 1.f;
        co = n.y ? n.out[0] : 0.f;
        ci = n.in ? n.in[0] : 1.f;
#pragma unroll
        for (int k = 0; k < NP; ++k)
        {
            bool on;
            const int c = piece(width, k, on);
            x[k] = reinterpret_cast<const float4*>(n.x)[c];
            y[k] = reinterpret_cast<const float4*>(y_or_x)[c];
            w[k] = reinterpret_cast<const float4*>(n.w)[c];
        }
        asm volatile("" ::: "memory"); // (what is requested next does not go in front)
    }
    __device__ __forceinline__ void finish(const StackRowNorm& n, int width, uint16_t* row, float* red, bool first)
    {
#pragma unroll
        for (int k = 0; k < NP; ++k)
        {
            bool on;
            const int c = piece(width, k, on);
            float4 v = x[k];
            if (n.y)
            {
                v = make_float4(fmaf(co, y[k].x, cm * v.x), fmaf(co, y[k].y, cm * v.y), fmaf(co, y[k].z, cm * v.z), fmaf(co, y[k].w, cm * v.w));
                if (first && on)
                    reinterpret_cast<float4*>(n.x_out)[c] = v;
            }
            x[k] = make_float4(ci * v.x, ci * v.y, ci * v.z, ci * v.w);
            const float ss = wave_sum(on ? sum_squares4<true>(x[k]) : 0.f);
            if ((threadIdx.x & 63) == 0)
                red[4 * k + (threadIdx.x >> 6)] = ss;
        }
        __syncthreads();
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < SUMS; ++i)
            ss += red[i];
        const float inv = 1.f / sqrtf(ss / (float) width + n.eps);
#pragma unroll
        for (int k = 0; k < NP; ++k)
        {
            bool on;
            const int c = piece(width, k, on);
            if (!on)
                continue;
            const uint2 h = make_uint2((uint32_t) f2bf(x[k].x * inv * w[k].x) | ((uint32_t) f2bf(x[k].y * inv * w[k].y) << 16),
                (uint32_t) f2bf(x[k].z * inv * w[k].z) | ((uint32_t) f2bf(x[k].w * inv * w[k].w) << 16));
            reinterpret_cast<uint2*>(row)[c] = h;
            if (first && n.h)
                reinterpret_cast<uint2*>(n.h)[c] = h;
        }
        __syncthreads();
    }
};

// A row in PARTS with a norm each, as group_rmsnorm_kernel: thread t has values t, t + 256, ... of a part, 64 lanes, 4 waves.  A part has up to 256 EACH values.
template <int NP, int PARTS>
struct PartsRow
{
    static constexpr int SUMS = 4 * PARTS, EACH = 4 * NP / PARTS;
    static_assert(EACH * PARTS == 4 * NP, "whole parts");
    float x[PARTS][EACH], w[PARTS][EACH];

    __device__ __forceinline__ static int place(int width, int g, int k, bool& on)
    {
        const int part = width / PARTS, i = threadIdx.x + 256 * k;
        on = i < part;
        return on ? g * part + i : 0;
    }
    __device__ __forceinline__ void request(const StackRowNorm& n, int width)
    {
#pragma unroll
        for (int g = 0; g < PARTS; ++g)
#pragma unroll
            for (int k = 0; k < EACH; ++k)
            {
                bool on;
                const int i = place(width, g, k, on);
                x[g][k] = n.x[i];
                w[g][k] = n.w[i];
            }
        asm volatile("" ::: "memory");
    }
    __device__ __forceinline__ void finish(const StackRowNorm& n, int width, uint16_t* row, float* red, bool first)
    {
#pragma unroll
        for (int g = 0; g < PARTS; ++g)
        {
#pragma unroll
            for (int k = 0; k < EACH; ++k)
            {
                bool on;
                place(width, g, k, on);
                x[g][k] = on ? x[g][k] : 0.f;
            }
            const float ss = wave_sum(sum_squares(x[g]));
            if ((threadIdx.x & 63) == 0)
                red[4 * g + (threadIdx.x >> 6)] = ss;
        }
        __syncthreads();
        const float4 r = reinterpret_cast<const float4*>(red)[threadIdx.x & (PARTS - 1)]; // (lane g has part g's root: one sequence of instructions instead of PARTS)
        const float root = 1.f / sqrtf((((r.x + r.y) + r.z) + r.w) / (float) (width / PARTS) + n.eps);
#pragma unroll
        for (int g = 0; g < PARTS; ++g)
        {
            const float inv = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, root), g));
#pragma unroll
            for (int k = 0; k < EACH; ++k)
            {
                bool on;
                const int i = place(width, g, k, on);
                if (!on)
                    continue;
                const float v = x[g][k] * inv;
                row[i] = f2bf(v * w[g][k]);
                if (first && n.h)
                    reinterpret_cast<uint16_t*>(n.h)[i] = f2bf(v * w[g][k]);
                if (first && n.h2)
                    reinterpret_cast<uint16_t*>(n.h2)[i] = f2bf(v * n.w2[i]);
            }
        }
        __syncthreads();
    }
};
template <int NP, int PARTS>
using LoneRow = typename std::conditional<PARTS == 0, StreamRow<NP>, PartsRow<NP, PARTS ? PARTS : 1>>::type;

} // namespace
} // namespace kernels
} // namespace tllm
