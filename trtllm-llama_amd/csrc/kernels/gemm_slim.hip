// Products of few rows on the LLaMA path: fp16, SmoothQuant int8, weight-only int8 / int4 weights through the weight-streaming main loop of
// gemm_slim_impl.h.  Short prompts and plain calls of 5 .. 31 rows (int4 weights 3 .. 31), generation steps of 5 .. 32 sequences with fp16 or
// weight-only weights (int4 3 .. 32; fp16 products without a norm ahead or SwiGLU behind from 3).  The epilogue has the rounding points of the tiles in gemm_mfma.hip.  The sums' order is not the
// streaming GEMV's, which serves fewer rows: a sequence's fp16 rows differ in their last bits with the number of rows beside it.
#include "gemm_slim_impl.h"
#include "kernels.h"
#include "launch_util.h"
#include "weight_layout.h"

namespace tllm
{
namespace kernels
{
using namespace dev;

namespace
{

// columns col0 .. col0 + 3 of one row
template <int WT>
__device__ __forceinline__ void finish4(const GemmParams& p, int row, int col0, const typename slim::Traits<WT>::acc_t& acc)
{
    constexpr bool SQ = WT == W_INT8_SQ;
    const float sr = SQ ? (p.per_token ? p.scale_row[row] : p.scale_row[0]) : 1.f;
#pragma unroll
    for (int e = 0; e < 4; ++e)
    {
        const int col = col0 + e;
        if (col >= p.N)
            continue;
        float v;
        if constexpr (SQ)
            v = (float) acc[e] * ((p.per_channel ? reinterpret_cast<const float*>(p.scale_col)[col] : reinterpret_cast<const float*>(p.scale_col)[0]) * sr);
        else if constexpr (WT == W_FP16)
            v = acc[e];
        else
            v = acc[e] * h2f(reinterpret_cast<const uint16_t*>(p.scale_col)[col]);
        const int64_t o = (int64_t) row * p.ldc + col;
        if (p.out_dtype == DT_HALF)
        {
            uint16_t y = f2h(v); // (what follows: the pointwise passes' own rounding points)
            if (p.residual)
                y = f2h(h2f(y) + h2f(reinterpret_cast<const uint16_t*>(p.residual)[o]));
            else if (p.silu_gate)
            {
                const float g = h2f(reinterpret_cast<const uint16_t*>(p.silu_gate)[o]);
                y = f2h(h2f(f2h(g / (1.f + __expf(-g)))) * h2f(y));
            }
            reinterpret_cast<uint16_t*>(p.c)[o] = y;
        }
        else if (SQ && p.out_dtype == DT_INT32)
            reinterpret_cast<int32_t*>(p.c)[o] = f2i32_rni_sat(v);
        else
            reinterpret_cast<float*>(p.c)[o] = v;
    }
}

// fp16, SmoothQuant int8
template <int WT, class S>
__global__ __launch_bounds__(S::waves * 64) void gemm_slim_kernel(const GemmParams p)
{
    extern __shared__ __attribute__((aligned(16))) char slim_lds[];
    constexpr int ES = WT == W_INT8_SQ ? 1 : 2;
    const int lane = threadIdx.x & 63, n0 = blockIdx.x * S::cols;
    slim::stream<WT, S>(slim_lds, reinterpret_cast<const char*>(p.w) + (int64_t) n0 * p.ldw, p.ldw, p.N - n0, p.K * ES,
        [&](int m) { return reinterpret_cast<const char*>(p.a) + (int64_t) (m < p.M ? m : p.M - 1) * p.lda * ES; },
        [&](int t, const typename slim::Traits<WT>::acc_t& acc) {
            const int row = 16 * t + (lane & 15), c = 4 * (lane >> 4);
            if (row < p.M && row < S::mt * S::cols && c < S::cols)
                finish4<WT>(p, row, n0 + c, acc);
        });
}

// weight-only int8 / int4
template <int WT, int MT, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void gemm_slim_woq_kernel(const GemmParams p)
{
    __shared__ __attribute__((aligned(16))) char lds[slim::lds_bytes<MT, WAVES>()];
    const int lane = threadIdx.x & 63;
    const int n0 = blockIdx.x * 16;
    const char* xrow[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
    {
        const int m = 16 * t + (lane & 15);
        xrow[t] = reinterpret_cast<const char*>(p.a) + (int64_t) (m < p.M ? m : p.M - 1) * p.lda * 2;
    }
    slim::product<WT, MT, WAVES>(lds, reinterpret_cast<const char*>(p.w) + (int64_t) n0 * p.ldw, p.ldw, p.N - n0, WT == W_INT4_WOQ ? p.K / 2 : p.K, xrow,
        [&](int t, const typename slim::Traits<WT>::acc_t& acc) {
            const int row = 16 * t + (lane & 15);
            if (row < p.M)
                finish4<WT>(p, row, n0 + 4 * (lane >> 4), acc);
        });
}

inline int launched()
{
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
    {
        set_error("gemm_slim launch failed: %s", hipGetErrorString(e));
        return -1;
    }
    return 0;
}

template <int WT>
int launch_stream(const GemmParams& p, hipStream_t stream)
{
    slim::pick_shape(p.M, p.N, 1, (int64_t) p.K * (WT == W_INT8_SQ ? 1 : 2), false, launch_util::device_cus(), [&](auto shape) {
        using S = decltype(shape);
        launch_util::ensure_dynamic_lds(reinterpret_cast<const void*>(&gemm_slim_kernel<WT, S>), S::lds_bytes);
        hipLaunchKernelGGL((gemm_slim_kernel<WT, S>), dim3((p.N + S::cols - 1) / S::cols), dim3(S::waves * 64), S::lds_bytes, stream, p);
    });
    return launched();
}

template <int WT, int MT, int WAVES>
int go(const GemmParams& p, hipStream_t stream)
{
    hipLaunchKernelGGL((gemm_slim_woq_kernel<WT, MT, WAVES>), dim3((p.N + 15) / 16), dim3(WAVES * 64), 0, stream, p);
    return launched();
}

template <int WT>
int launch_wt(const GemmParams& p, hipStream_t stream)
{
    // (two row tiles: 12288 x 4096 weight-only int8 at 19 rows 26.0 us on 4 waves, 27.9 on 8; 4096 x 11008 26.8 and 21.1)
    const bool many = (p.N + 15) / 16 * 4 >= launch_util::device_cus() * 5;
    if (p.M <= 16)
        return many ? go<WT, 1, 4>(p, stream) : go<WT, 1, 8>(p, stream);
    return many ? go<WT, 2, 4>(p, stream) : go<WT, 2, 8>(p, stream);
}

} // namespace

// Rows from which this form is the quicker one (the streaming GEMV's time grows with the rows: dot products on the vector pipe, and LDS for
// every row's activations).  Cold weights, us at 4 / 5 / 8 rows by the GEMV and at 8 here (timed with bfloat16): fp16 4096 x 4096 9.3 / 11.5 /
// 12.0, 7.8; fp16 4096 x 11008 19.9 / 36.8 / 39.3, 18.7 (from 3 rows where there is nothing but the product to do: session.cpp's gemv); at 9
// here: SmoothQuant 4096 x 11008 12.9 / 15.5 / 16.5, 12.7; int8 weights 12288 x 4096 16.0 / 28.6 / 28.9, 16.8; int4 weights 12288 x 4096 at
// 2 / 4 / 5 rows 16.4 / 31.5 / 195, 15.0.
int gemm_slim_rows(int wtype)
{
    return wtype == W_INT4_WOQ ? 3 : 5;
}

bool gemm_slim_serves(const GemmParams& p)
{
    if (p.wtype != W_FP16 && p.wtype != W_INT8_SQ && p.wtype != W_INT8_WOQ && p.wtype != W_INT4_WOQ)
        return false;
    const int a_es = p.wtype == W_INT8_SQ ? 1 : 2;
    if (p.M < 1 || p.M > 32 || p.N < 1 || p.K < 1 || ((p.residual || p.silu_gate) && p.out_dtype != DT_HALF))
        return false;
    // 16-byte loads of both operands; 32-bit offsets of a workgroup's W rows
    if ((reinterpret_cast<uintptr_t>(p.a) & 15) || ((p.lda * a_es) & 15) || (reinterpret_cast<uintptr_t>(p.w) & 15) || (p.ldw & 15) || p.ldw > (1 << 26))
        return false;
    if ((p.K * a_es) % 16 || (p.wtype == W_INT8_WOQ && p.K % 16) || (p.wtype == W_INT4_WOQ && p.K % 32))
        return false;
    return p.out_dtype == DT_HALF || p.out_dtype == DT_FLOAT || (p.out_dtype == DT_INT32 && p.wtype == W_INT8_SQ);
}

// 0: launched, -1: launch error, 1: not served.  residual and silu_gate share c's rows; c may be the residual itself
int launch_gemm_slim(const GemmParams& p, hipStream_t stream)
{
    if (!gemm_slim_serves(p))
        return 1;
    switch (p.wtype)
    {
    case W_FP16: return launch_stream<W_FP16>(p, stream);
    case W_INT8_SQ: return launch_stream<W_INT8_SQ>(p, stream);
    case W_INT8_WOQ: return launch_wt<W_INT8_WOQ>(p, stream);
    default: return launch_wt<W_INT4_WOQ>(p, stream);
    }
}

} // namespace kernels
} // namespace tllm
