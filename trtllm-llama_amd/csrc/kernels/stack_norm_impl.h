// A lone token's normed row, formed by the workgroups that read it (stack_kernels.h, StackRowNorm): shared by its products (stack_gemm.hip) and its
// router's logits (stack_moe.hip).  Everything has internal linkage.
#pragma once
#include "dev_utils.h"
#include "stack_kernels.h"

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

// A workgroup of 4 waves; wave q has the q-th quarter of the row, NP pieces of 4 values a lane, so that up to 4 parts with a norm each end where a wave does, and 8 (whole
// pieces of the wave each) where half of its pieces do.
template <int NP>
struct LoneRow
{
    float4 x[NP], y[NP], w[NP];
    float cm, co, ci;

    __device__ __forceinline__ static int piece(int width, int k, bool& on)
    {
        const int quarter = width >> 4, i = (threadIdx.x & 63) + 64 * k;
        on = i < quarter;
        return (int) (threadIdx.x >> 6) * quarter + (on ? i : 0);
    }
    // all loads, without a branch that they would wait behind; ahead of the operands that they are to arrive before
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
    // row: LDS [width], the normed row in bfloat16; red: LDS [4].  first: this workgroup also leaves what later launches read.
    __device__ __forceinline__ void finish(const StackRowNorm& n, int width, uint16_t* row, float* red, bool first)
    {
        const int wid = threadIdx.x >> 6;
        float ss = 0.f, front = 0.f; // front: of the first half of the pieces
#pragma unroll
        for (int k = 0; k < NP; ++k)
        {
            bool on;
            const int c = piece(width, k, on);
            if (k == NP / 2)
                front = ss, ss = 0.f;
            float4 v = x[k];
            if (n.y)
            {
                v = make_float4(fmaf(co, y[k].x, cm * v.x), fmaf(co, y[k].y, cm * v.y), fmaf(co, y[k].z, cm * v.z), fmaf(co, y[k].w, cm * v.w));
                if (first && on)
                    reinterpret_cast<float4*>(n.x_out)[c] = v;
            }
            v = make_float4(ci * v.x, ci * v.y, ci * v.z, ci * v.w);
            x[k] = v;
            ss += on ? v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w : 0.f;
        }
        float inv_front, inv;
        if (n.groups == 8)
        {
            inv_front = 1.f / sqrtf(wave_sum(front) / (float) (width >> 3) + n.eps);
            inv = 1.f / sqrtf(wave_sum(ss) / (float) (width >> 3) + n.eps);
        }
        else
        {
            ss = wave_sum(front + ss);
            if ((threadIdx.x & 63) == 0)
                red[wid] = ss;
            __syncthreads();
            ss = n.groups == 4 ? red[wid] : n.groups == 2 ? red[wid & 2] + red[wid | 1] : (red[0] + red[1]) + (red[2] + red[3]);
            inv_front = inv = 1.f / sqrtf(ss / (float) (width / n.groups) + n.eps);
        }
#pragma unroll
        for (int k = 0; k < NP; ++k)
        {
            bool on;
            const int c = piece(width, k, on);
            const float by = k < NP / 2 ? inv_front : inv;
            auto normed = [&](const float4& s) {
                return make_uint2((uint32_t) f2bf(x[k].x * by * s.x) | ((uint32_t) f2bf(x[k].y * by * s.y) << 16),
                    (uint32_t) f2bf(x[k].z * by * s.z) | ((uint32_t) f2bf(x[k].w * by * s.w) << 16));
            };
            if (!on)
                continue;
            const uint2 h = normed(w[k]);
            reinterpret_cast<uint2*>(row)[c] = h;
            if (first && n.h)
                reinterpret_cast<uint2*>(n.h)[c] = h;
            if (first && n.h2)
                reinterpret_cast<uint2*>(n.h2)[c] = normed(reinterpret_cast<const float4*>(n.w2)[c]);
        }
        __syncthreads();
    }
};

} // namespace
} // namespace kernels
} // namespace tllm
