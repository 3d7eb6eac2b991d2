// Products of few rows, C[m, n] = sum_k A[m, k] * W[n, k] with M <= 32, bound by the weights' way through the memory system: the main loop shared
// by the stack engine's bfloat16 products (stack_gemm.hip) and the LLaMA path's fp16 / int8 / weight-only ones (gemm_slim.hip).
//
// A workgroup owns 16 rows of W (columns of C) and all M <= 16 * MT rows of A; its waves split K: 256-byte block j of every W row belongs to wave
// j mod WAVES, so that the waves together walk 1 or 2 KiB runs of each row.  A wave requests a block as 4 rows x 256 contiguous bytes
// per instruction (loads in the MFMA fragment's own geometry, 16 rows x 64 bytes, touch every 128-byte line twice), D blocks ahead in
// registers, turns it around in a private 4 KiB of LDS (16-byte pieces XOR-ed with the row: the row-wise writes and the fragment reads are
// free of bank conflicts) and feeds v_mfma_*_16x16: W is the A operand, the activation rows the B operand, read straight from the
// cache in fragment geometry (every workgroup reads the same few rows).  No barrier in the main loop - LDS operations of one wave
// complete in order; the waves' partial sums meet in LDS once at the end, in a fixed order.
//
// Time hardly depends on M.  Measured (us, bfloat16, cold weights, back to back; N x K; in brackets what they took as dot products on
// the vector pipe, M = 8, and as 128 x 128 register-staged tiles)
// M = 8, 9, 31:   2048 x 2048 6.6, 6.5, 8.7 (12.3, 131, 137)    4096 x 11008 20.8, 20.8, 31.6 (39.5, 680, 687)
//                 22016 x 4096 34.1, 34.6, 60.9 = 5.3 TB/s at 8 rows (62.4, 266, 273)    32000 x 2048 30.3, 30.5, 44.5 (51.5, 158, 165)
// What the launch shapes below are chosen from (M = 8): 4 waves, one block ahead: 32000 x 2048 28.8, 22016 x 4096 32.4, 11008 x 2048 12.0 against
// 35.7, 39.3, 15.0 for 8 waves, two ahead; 4096 x 11008 24.4 against 19.4, 2048 x 5504 12.5 against 9.1, 6144 x 2048 8.6 against 10.1: once
// there are more workgroups than fill the chip, more requests in flight per workgroup only thrash.  Blocks of 128, 512 or 1024 bytes and 32 rows
// of W per workgroup measured between 3 % better and 60 % worse over the same shapes.
//
// Byte geometry: a k-step is 64 bytes of W per row, lane l supplies row l & 15, piece l >> 4.  bfloat16, fp16: v_mfma_f32_16x16x32; int8:
// v_mfma_i32_16x16x64_i8 (exact); weight-only int8 / int4: the 16 bytes hold 16 / 32 weights of consecutive k, dequantised to fp16
// (exactly) behind the fragment read and consumed by 2 / 4 fp16 MFMAs.
#pragma once
#include "dev_utils.h"
#include "kernels.h"
#include <type_traits>

namespace tllm
{
namespace dev
{
namespace slim
{
using namespace kernels;
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int CB = 256;                                          // bytes of a W row per block
constexpr int PPR = CB / 16, RPI = 64 / PPR, NL = 16 / RPI, KS = CB / 64; // pieces per row, rows per request, requests and k-steps per block

template <int WT>
struct Traits
{
    using acc_t = typename std::conditional<WT == W_INT8_SQ, i32x4, f32x4>::type;
    static constexpr int XP = WT == W_INT8_WOQ ? 2 : (WT == W_INT4_WOQ ? 4 : 1); // 16-byte pieces of a row of A per piece of W
};

// u8 (q + 128) x 8 -> 8 fp16 (q, exactly)
__device__ __forceinline__ uint4 deq_u8x8(uint32_t w0, uint32_t w1)
{
    const uint32_t magic = 0x64646464u;
    const h2_t bias = {(_Float16) 1152.f, (_Float16) 1152.f};
    return make_uint4(h2_as_u32(u32_as_h2(__builtin_amdgcn_perm(magic, w0, 0x04010400u)) - bias), h2_as_u32(u32_as_h2(__builtin_amdgcn_perm(magic, w0, 0x04030402u)) - bias),
        h2_as_u32(u32_as_h2(__builtin_amdgcn_perm(magic, w1, 0x04010400u)) - bias), h2_as_u32(u32_as_h2(__builtin_amdgcn_perm(magic, w1, 0x04030402u)) - bias));
}
// 8 nibbles of a word (weight_layout.h) -> 8 fp16 (q, exactly) in the order of k
__device__ __forceinline__ uint4 deq_u4x8(uint32_t w)
{
    const uint32_t m = 0x64006400u, w8 = w >> 8;
    const h2_t b0 = {(_Float16) 1032.f, (_Float16) 1032.f}, s1 = {(_Float16) 0.0625f, (_Float16) 0.0625f}, b1 = {(_Float16) -72.f, (_Float16) -72.f};
    return make_uint4(h2_as_u32(u32_as_h2((w & 0x000f000fu) | m) - b0), h2_as_u32(u32_as_h2((w & 0x00f000f0u) | m) * s1 + b1),
        h2_as_u32(u32_as_h2((w8 & 0x000f000fu) | m) - b0), h2_as_u32(u32_as_h2((w8 & 0x00f000f0u) | m) * s1 + b1));
}

template <int WT>
__device__ __forceinline__ void mma(typename Traits<WT>::acc_t& acc, const uint4& w, const uint4* x)
{
    if constexpr (WT == W_INT8_SQ)
    {
        const i32x4 a = {(int) w.x, (int) w.y, (int) w.z, (int) w.w}, b = {(int) x[0].x, (int) x[0].y, (int) x[0].z, (int) x[0].w};
        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, acc, 0, 0, 0);
    }
    else if constexpr (WT == W_BF16)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, x[0]), acc, 0, 0, 0);
    else if constexpr (WT == W_FP16)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w), __builtin_bit_cast(f16x8, x[0]), acc, 0, 0, 0);
    else if constexpr (WT == W_INT8_WOQ)
    {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, deq_u8x8(w.x, w.y)), __builtin_bit_cast(f16x8, x[0]), acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, deq_u8x8(w.z, w.w)), __builtin_bit_cast(f16x8, x[1]), acc, 0, 0, 0);
    }
    else
    {
        const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, deq_u4x8(ws[i])), __builtin_bit_cast(f16x8, x[i]), acc, 0, 0, 0);
    }
}

// bytes of LDS: a wave's block of W (the partial sums reuse the room: one 16 x 16 tile is 1 KiB)
template <int MT, int WAVES>
constexpr int lds_bytes()
{
    return WAVES * (16 * CB > MT * 1024 ? 16 * CB : MT * 1024);
}

// w: the workgroup's first row of W, ldw bytes apart (16 ldw < 2^32), `rows` of them exist (>= 1; the others repeat the last one and their results are
// not to be stored).  wbytes: bytes of a W row that hold weights, a multiple of 16.  xrow[t]: this lane's row 16 t + (lane & 15) of A (a valid
// row also where that one does not exist), wbytes * XP bytes.  At the end wave t calls finish(t, acc), acc[e] = C[16 t + (lane & 15)]
// [first row + 4 (lane >> 4) + e].
template <int WT, int MT, int D, int WAVES, class Finish>
__device__ __forceinline__ void product(char* lds, const char* w, int64_t ldw, int rows, int wbytes, const char* const (&xrow)[MT], Finish finish)
{
    using T = Traits<WT>;
    using acc_t = typename T::acc_t;
    constexpr int XP = T::XP;
    
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, g4 = lane >> 4;
    char* mine = lds + wid * (16 * CB);
    const int lr = lane / PPR, lp = lane % PPR;

    // this lane's part of a block request
    uint32_t woff[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i)
    {
        const int r = RPI * i + lr;
        woff[i] = (uint32_t) ((r < rows ? r : rows - 1) * ldw) + lp * 16;
    }
    const int nblk = (wbytes + CB - 1) / CB;
    uint4 wv[D][NL], xv[D][MT][KS * XP];
    auto request = [&](int d, int q) {
        const int base = q * CB;
        const bool w_in = base + lp * 16 < wbytes;
#pragma unroll
        for (int i = 0; i < NL; ++i)
            wv[d][i] = w_in ? ld_nt16(w + base + woff[i]) : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int s = 0; s < KS; ++s)
        {
            const int at = base + s * 64 + g4 * 16; // of the W row
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int u = 0; u < XP; ++u)
                    xv[d][t][s * XP + u] = at < wbytes ? *reinterpret_cast<const uint4*>(xrow[t] + (int64_t) at * XP + u * 16) : make_uint4(0, 0, 0, 0);
        }
    };

    acc_t acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
        acc[t] = acc_t{0, 0, 0, 0};

    auto consume = [&](int d) {
#pragma unroll
        for (int i = 0; i < NL; ++i)
        {
            const int r = RPI * i + lr;
            *reinterpret_cast<uint4*>(mine + r * CB + ((lp ^ (r & 15)) << 4)) = wv[d][i];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); // (the reads below are of other lanes' pieces)
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int s = 0; s < KS; ++s)
        {
            const uint4 wf = *reinterpret_cast<const uint4*>(mine + r16 * CB + (((s * 4 + g4) ^ r16) << 4));
#pragma unroll
            for (int t = 0; t < MT; ++t)
                mma<WT>(acc[t], wf, &xv[d][t][s * XP]);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };

    // Blocks wid, wid + WAVES, ...: `count` of them.  While at least 2 D are left every request of a round is certain - a request that might not
    // be made would have the compiler wait as if it had not been, with the ring drained each time.
    const int count = (nblk - wid + WAVES - 1) / WAVES;
    auto block = [&](int i) { return wid + i * WAVES; };
    if (count >= D)
    {
#pragma unroll
        for (int d = 0; d < D; ++d)
            request(d, block(d));
        int i = 0;
        for (; i + 2 * D <= count; i += D)
#pragma unroll
            for (int d = 0; d < D; ++d)
            {
                consume(d);
                request(d, block(i + D + d));
            }
#pragma unroll
        for (int d = 0; d < D; ++d)
        {
            consume(d);
            if (i + D + d < count)
                request(d, block(i + D + d));
        }
#pragma unroll
        for (int d = 0; d < D - 1; ++d)
            if (i + D + d < count)
                consume(d);
    }
    else
    {
#pragma unroll
        for (int d = 0; d < D - 1; ++d)
            if (d < count)
                request(d, block(d));
#pragma unroll
        for (int d = 0; d < D - 1; ++d)
            if (d < count)
                consume(d);
    }

    // the waves' sums meet: [wave][tile][lane]
    __syncthreads();
    acc_t* red = reinterpret_cast<acc_t*>(lds);
#pragma unroll
    for (int t = 0; t < MT; ++t)
        red[(wid * MT + t) * 64 + lane] = acc[t];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < MT; ++t)
        if (t == wid)
        {
            acc_t v = red[t * 64 + lane];
#pragma unroll
            for (int k = 1; k < WAVES; ++k)
                v += red[(k * MT + t) * 64 + lane];
            finish(t, v);
        }
}

} // namespace slim
} // namespace dev
} // namespace tllm
