// The choice of experts inside a wave (stack_kernels.h, StackMoeParams), shared by the router's launches (stack_moe.hip) and a lone token's expert
// products, which choose for themselves (stack_gemm.hip).
#pragma once
#include "dev_utils.h"
#include "stack_kernels.h"

namespace tllm
{
namespace kernels
{
using namespace dev;

// the lane that holds the largest value of the wave, the lowest index among equals; every lane gets (value, index).  The maximum goes
// through DPP moves, and a lane that holds it alone gives its index by a lane read: a twelve-shuffle tree costs twice the time of a choice.
__device__ __forceinline__ void wave_argmax(float& v, int& idx)
{
    const float m = wave_max(v);
    const uint64_t at = __ballot(v == m);
    if (__popcll(at) == 1)
        idx = __builtin_amdgcn_readlane(idx, (int) __builtin_ctzll(at));
    else
    {
        int best = v == m ? idx : 0x7fffffff;
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1)
        {
            const int o = __shfl_xor(best, d, 64);
            best = o < best ? o : best;
        }
        idx = best;
    }
    v = m;
}

// select_token (stack_moe.hip) for up to LONE_OUT outputs, an output per lane and everything in registers: the same values in the same order.
// z: this lane's logit, bias added; c: its correction.  Lane k < top gets choice k and its weight.
constexpr int LONE_OUT = 64;
struct Chosen
{
    int output;
    float weight;
};
__device__ __forceinline__ Chosen choose_in_wave(const StackMoeParams& p, float z, float c, int lane)
{
    const int NE = p.experts + p.identity;
    const bool on = lane < NE;
    float s;
    if (p.score == ROUTE_SIGMOID)
        s = 1.f / (1.f + expf(-z));
    else
    {
        const float mx = wave_max(on ? z : -INFINITY);
        const float x = on ? expf(z - mx) : 0.f;
        const float inv = 1.f / wave_sum(x);
        s = x * inv;
    }
    c = on ? c + s : -INFINITY;
    const int GC = p.group_count, GS = NE / GC;
    if (GC > 1 && p.group_keep < GC)
    {
        // lane g < GC: its group's largest choice value
        float gv = -INFINITY;
        for (int g = 0; g < GC; ++g)
        {
            const float m = wave_max(on && lane / GS == g ? c : -INFINITY);
            gv = lane == g ? m : gv;
        }
        uint64_t kept = 0;
        for (int k = 0; k < p.group_keep; ++k)
        {
            const bool open = lane < GC && !(kept >> lane & 1);
            float bv = open ? gv : -INFINITY;
            int bi = open ? lane : 0x7fffffff;
            wave_argmax(bv, bi);
            kept |= bi < GC ? (uint64_t) 1 << bi : 0;
        }
        if (on && !(kept >> (lane / GS) & 1))
            c = -INFINITY;
    }
    float mine = 0.f, total = 0.f;
    int chosen = 0;
    for (int k = 0; k < p.top; ++k)
    {
        const bool open = c > -INFINITY; // (not a NaN either)
        float bv = open ? c : -INFINITY;
        int bi = open ? lane : 0x7fffffff;
        wave_argmax(bv, bi);
        if (bi >= NE) // fewer choosable outputs than `top`: the place stays empty (weight 0 on the last one)
            bi = NE - 1, bv = -INFINITY;
        const float got = bv == -INFINITY ? 0.f : __shfl(s, bi, 64);
        total += got;
        if (lane == k)
        {
            mine = got;
            chosen = bi;
        }
        if (lane == bi)
            c = -INFINITY;
    }
    return {chosen, (p.normalize ? mine / (total + 1e-20f) : mine) * p.scale};
}

} // namespace kernels
} // namespace tllm
