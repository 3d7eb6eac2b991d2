// SmoothQuant int8 and fp16 products of many rows on the 256 x 256 tiles of gemm_wide_impl.h, or its tiles of 128 rows:  C[m,n] = float(sum_k X[m,k] * W[n,k]) * (s_col[n] * s_row[m])
// (A10: K/cutlass_kernels/int8_gemm/int8_gemm_template.h:56-172, epilogue K/cutlass_extensions/.../epilogue_per_row_per_col_scale.h:279-347 - exact int32
// accumulation, one fp32 scale product; A7 P/gemmPlugin/gemmPlugin.cpp:121-190 in fp16), and the two int8 products of an MLP with SwiGLU and the static quantiser behind them.
#include "gemm_wide_impl.h"

namespace tllm
{
namespace kernels
{

extern void* gemm_clock_probe; // gemm_sqp.hip (microbench hook)

// 0 launched, -1 launch error, 1 not served
int launch_gemm_wide(const GemmParams& p, hipStream_t stream)
{
    if (p.M < 32)
        return 1;
    if (wide::serves<W_FP16>(p))
        return wide::launch<W_FP16>(p, stream);
    return wide::serves<W_INT8_SQ>(p) ? wide::launch<W_INT8_SQ>(p, stream) : 1;
}

bool gemm_rows128_serves(const GemmParams& p)
{
    return p.M >= 32 && (p.wtype == W_FP16 ? wide::serves<W_FP16>(p) : !p.w2 && wide::serves<W_INT8_SQ>(p));
}
template <int WT>
static int launch_rows128_type(const GemmParams& p, bool wide_cols, hipStream_t stream)
{
    return wide_cols ? wide::launch_row128_out<WT, wide::OUT_HALF, false, 2, 4, 2, 2, 3, true>(p, stream)
                     : wide::launch_row128_out<WT, wide::OUT_HALF, false, 2, 4, 2, 1, 4, false>(p, stream);
}
// tiles of 128 x 128, or of 128 x 256: 0 launched, -1 launch error, 1 not served
int launch_gemm_rows128(const GemmParams& p_in, bool wide_cols, hipStream_t stream)
{
    if (!gemm_rows128_serves(p_in))
        return 1;
    GemmParams p = p_in;
    p.clock_probe = gemm_clock_probe;
    return p.wtype == W_FP16 ? launch_rows128_type<W_FP16>(p, wide_cols, stream) : launch_rows128_type<W_INT8_SQ>(p, wide_cols, stream);
}

// the time in K-tiles of a 256 x 256 tile (wide::cost) is less than `other`, and the product is served
bool gemm_wide_beats(const GemmParams& p, double other)
{
    const bool fp16 = p.wtype == W_FP16;
    return p.M >= 32 && (fp16 ? wide::serves<W_FP16>(p) : wide::serves<W_INT8_SQ>(p)) && wide::cost(p, fp16 ? 2 : 1) < other;
}

} // namespace kernels
} // namespace tllm
