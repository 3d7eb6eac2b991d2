// The short causal convolution of the recurrent layers for a step of one row: each workgroup of the recurrence's step kernel forms the channels that it reads, instead
// of a launch in front of it, which costs its start and 3.6 - 3.8 us for a few loads a thread: the raw inputs are requested behind the state, whose way takes longer.
// us, convolution + step and here: 64 heads of 128 x 64 in 8 groups 3.8 + 4.5, 5.1; 8 delta heads of 128 x 128 3.7 + 6.0, 7.0.  A header, so that stack_ssm.hip and stack_delta.hip share one source; everything has internal linkage.
//
// A sequence's raw inputs lie in a ring of `taps` rows, row q of it (counted as they are fed) in row q mod taps.  A row reads the taps - 1 in front of it and writes its own:
// a row that nobody reads in this launch, so heads that share channels may all read them while one of them writes.
#pragma once
#include "dev_utils.h"

namespace tllm
{
namespace kernels
{
namespace
{

template <int DT, int TAPS>
struct ConvStep
{
    float old[TAPS - 1], now, w[TAPS], bias;

    // channel c; in: the row's first channel; ring: the slot's
    __device__ __forceinline__ void request(const void* in, const float* ring, const float* conv_w, const float* conv_b, int channels, int fed, int c)
    {
        static_assert(TAPS == 4, "weights in one piece");
#pragma unroll
        for (int j = 0; j < TAPS - 1; ++j)
        {
            const int q = fed - (TAPS - 1) + j;
            old[j] = q >= 0 ? ring[(int64_t) (q % TAPS) * channels + c] : 0.f;
        }
        if constexpr (DT == DT_BF16)
            now = dev::bf2f(reinterpret_cast<const uint16_t*>(in)[c]);
        else
            now = reinterpret_cast<const float*>(in)[c];
        const float4 x = reinterpret_cast<const float4*>(conv_w)[c];
        w[0] = x.x, w[1] = x.y, w[2] = x.z, w[3] = x.w;
        bias = conv_b ? conv_b[c] : 0.f;
    }
    // as the launch of its own leaves it: added up in its order, rounded to the element type
    __device__ __forceinline__ float value() const
    {
        float acc = bias;
#pragma unroll
        for (int j = 0; j < TAPS - 1; ++j)
            acc = fmaf(w[j], old[j], acc);
        acc = fmaf(w[TAPS - 1], now, acc);
        acc = acc / (1.f + expf(-acc));
        return DT == DT_BF16 ? dev::bf2f(dev::f2bf(acc)) : acc;
    }
};

// out[i] = channel channel_of(i) of the row, i < n; own(i): this workgroup writes its raw input into the ring.  Two channels of a thread are under way at a time.
template <int DT, class Channel, class Own>
__device__ __forceinline__ void conv_step(const void* in, float* ring, const float* conv_w, const float* conv_b, int channels, int fed, int n, float* out, Channel channel_of, Own own)
{
    constexpr int TAPS = 4, AT_ONCE = 2;
    for (int i0 = threadIdx.x; i0 < n; i0 += AT_ONCE * blockDim.x)
    {
        ConvStep<DT, TAPS> s[AT_ONCE];
#pragma unroll
        for (int u = 0; u < AT_ONCE; ++u)
        {
            const int i = i0 + u * blockDim.x;
            s[u].request(in, ring, conv_w, conv_b, channels, fed, channel_of(i < n ? i : i0));
        }
#pragma unroll
        for (int u = 0; u < AT_ONCE; ++u)
        {
            const int i = i0 + u * blockDim.x;
            if (i >= n)
                break;
            out[i] = s[u].value();
            if (own(i))
                ring[(int64_t) (fed % TAPS) * channels + channel_of(i)] = s[u].now;
        }
    }
}

} // namespace
} // namespace kernels
} // namespace tllm
