// Products of few rows, C[m, n] = sum_k A[m, k] * W[n, k] with M <= 32, bound by the weights' way through the memory system: the main loops shared
// by the stack engine's bfloat16 products (stack_gemm.hip) and the LLaMA path's fp16 / int8 / weight-only ones (gemm_slim.hip).
//
// A workgroup owns CW rows of W (columns of C) and all M <= 16 * MT rows of A; its waves split K: block j of every W row belongs to wave j mod WAVES.
// A block is 16 fragment rows of 256 bytes (loads in the MFMA fragment's own geometry, 16 rows x 64 bytes, touch every 128-byte line twice):
// CW = 16 rows of W, or one 512-byte run of each of 8.  It is read back from a private piece of LDS, its 16-byte pieces XOR-ed with the row
// so that neither side has bank conflicts, and feeds v_mfma_*_16x16: W is the A operand, the activation rows the B operand.  No barrier in the
// main loop; the waves' partial sums meet in LDS once at the end, in a fixed order.
//
// stream(): both operands come by LDS-DMA, D blocks ahead in a ring of the wave's own, so that a lane holds no block in registers (40 .. 50
// VGPRs, and what is in flight per CU is what its LDS holds) and rows of A are requested once per workgroup, 4 rows x 256 bytes an instruction.
// product(): a block ahead in registers, A straight from the cache in fragment geometry; for weight-only types, whose rows of A are 2 and 4 times
// as long as W's, and for grouped products whose groups have few rows (groups_by_registers).
//
// Time hardly depends on M up to 8 rows.  Measured, cold weights, back to back, us, bfloat16, N x K at 8 / 16 / 31 rows, in brackets the register form:
//   2048 x 2048 4.0 / 5.0 / 6.1 (5.3 / 6.1 / 7.5)    2048 x 5504 7.5 / 9.0 / 11.2 (9.1 / 10.6 / 15.1)    4352 x 2048 6.7 / 7.2 / 8.9 (9.5 / 11.1 / 13.5)
//   11008 x 2048 10.8 / 11.2 / 13.5 (12.1 / 13.6 / 18.6)    4096 x 4096 7.8 / 8.9 / 10.5 (9.1 / 9.9 / 12.9)    4096 x 11008 18.7 / 19.9 / 23.2 (19.6 / 21.6 / 28.4)
//   22016 x 4096 30.3 = 5.9 TB/s / 34.2 / 44.1 (32.1 / 39.5 / 59.5)    32000 x 2048 24.6 / 27.4 / 35.7 (28.7 / 31.8 / 43.7)
// The launch shapes (Shape below) for long rows are chosen from these: few columns want narrow workgroups (2048 x 2048, 8 rows: 8 columns 4.0, 16 columns 4.6 us);
// up to a workgroup per CU 8 waves (4096 x 4096 7.8 against 8.5 for 4); more workgroups than CUs fewer waves of fewer blocks, as requests
// beyond what fills the memory system only thrash (4352 x 2048, 8 rows: 8 columns by 4 waves one block ahead 6.7, 16 columns by 4 waves 7.2, by 8 waves
// 7.7; 31 rows by 2 waves 8.9, by 4 waves 10.5), but long rows still 4 (22016 x 4096, 16 rows: 34.2 against 40.2 for 2).
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

constexpr int CB = 256;                                                   // bytes of a fragment row per block
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

// Launch shape of stream(): `cols` columns of C per workgroup of `waves` waves, `depth` blocks ahead, 4 * xi fragment rows of A requested per block.
template <int COLS, int WAVES_, int DEPTH, int XI>
struct Shape
{
    static constexpr int cols = COLS, waves = WAVES_, depth = DEPTH, xi = XI, mt = XI > 4 ? 2 : 1;
    static constexpr int ring = DEPTH * (16 + 4 * XI) * CB; // bytes of LDS per wave (the partial sums reuse the room: a 16 x 16 tile is 1 KiB)
    static_assert((COLS == 16 || (COLS == 8 && XI == 4)) && ring >= mt * 1024, "narrow workgroups hold up to 8 rows of A");
    static constexpr int lds_bytes = WAVES_ * ring;
};
// calls f with the shape for m rows, n columns of `products` products and rows of W of `wbytes` bytes; grouped: a workgroup looks up its product first.
// Rows below 4 KiB end within a few blocks a wave: there what counts is how many workgroups a CU holds, so two waves, and from four workgroups per CU on
// a single block ahead; us at 8 rows, in brackets the shapes for longer rows: 32000 x 64 5.1 (14.4), x 512 9.0 (15.4), x 1792 21.6 (25.0), 11008 x 256
// 4.7 (7.7), x 1792 9.7 (12.0), 2048 x 64 3.8 (4.3); at 16 rows 32000 x 256 6.8 (9.5).  Rows of 4 KiB, each on the same memory channels as the one
// before, want 8 columns in 512-byte runs up to 8 rows: 8192 x 2048 9.9 (16 columns 11.0), 32000 x 2048 at 2 rows 24.9 (27.4).  31 rows by 2 waves two blocks ahead
// fill a third of a CU's LDS: beyond three workgroups per CU one block ahead, 13056 x 128 5.1 (7.3), 16384 x 2048 18.3 (23.5), x 11008 84 (99), of
// long rows up to four per CU (22016 x 11008 126, 121 with two).
template <class F>
inline auto pick_shape(int m, int64_t n, int64_t products, int64_t wbytes, bool grouped, int cus, F f)
{
    const int64_t wgs = (n + 15) / 16 * products;
    const bool many = wgs > cus, crowd = wgs >= 4 * cus, brief = wbytes <= 4096;
    if (m <= 8)
    {
        if (crowd && (grouped ? brief : wbytes < 4096))
            return f(Shape<16, 2, 1, 2>());
        if (wbytes <= 512 || (many && (grouped ? wbytes <= 1024 : wbytes < 4096)))
            return f(Shape<16, 2, 2, 2>());
        if (wgs * 2 <= cus)
            return f(Shape<8, 4, 2, 4>());
        if (!many)
            return f(Shape<16, 8, 2, 2>());
        return brief && !grouped ? f(Shape<8, 4, 1, 4>()) : f(Shape<16, 4, 2, 2>());
    }
    if (m <= 16)
    {
        if (crowd && wbytes <= 1024)
            return f(Shape<16, 2, 1, 4>());
        return many && brief ? f(Shape<16, 2, 2, 4>()) : f(Shape<16, 4, 2, 4>());
    }
    if (wgs > 3 * cus && (brief || wgs <= 4 * cus))
        return f(Shape<16, 2, 1, 8>());
    return many ? f(Shape<16, 2, 2, 8>()) : f(Shape<16, 4, 2, 8>());
}
// Whether grouped products of up to m rows go through product(), 4 waves: a group mostly has a row or two of them, and stream() brings all 8, 16 or
// 32 rows of A that its shape has room for to LDS for each.  32 groups, 4 of them per token, weights cold, us, in brackets stream(); N x K at 8 tokens:
// 2816 x 256 10.7 (17.8), x 1024 21.1 (24.5), x 2048 42.1 (45.2), x 3072 54.6 (53.2); at 16 tokens 2816 x 512 15.6 (21.3), x 2048 55.3 (61.4), x 4096
// 100 (100); at 31 tokens 1408 x 512 14.3 (17.2), x 2048 41.9 (43.2), x 4096 64.6 (69.4).  Fewer workgroups, 704 x 2048 at 8 tokens 15.7 (15.0); 256 x 512 at 16
// and 31 4.9 (5.0), 6.7 (5.4), x 2048 10.9 (10.8), 12.6 (11.9).
inline bool groups_by_registers(int m, int64_t n, int64_t products, int64_t wbytes, int cus)
{
    const int64_t wgs = (n + 15) / 16 * products;
    return m > 8 ? wgs > 2 * cus : wgs >= 8 * cus && wbytes <= 4096;
}

// one LDS-DMA instruction: 64 lanes x 16 bytes -> LDS [lds_byte + lane * 16] (inline asm: for the builtin the compiler waits for everything in
// front of the next LDS read), from a wave-uniform base + a per-lane offset, past the caches' reuse; and from per-lane addresses
__device__ __forceinline__ void dma_nt(const char* base, uint32_t off, uint32_t lds_byte)
{
    uint32_t m0_keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt\n\ts_mov_b32 m0, %0" : "=&s"(m0_keep) : "v"(off), "s"(base), "s"(lds_byte) : "memory");
}
__device__ __forceinline__ void dma(const char* p, uint32_t lds_byte)
{
    uint32_t m0_keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0" : "=&s"(m0_keep) : "v"(p), "s"(lds_byte) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_requests()
{
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// The waves' sums meet: [wave][tile][lane]; wave t finishes tile t.  Tiles of 8 columns: run 1's sums lie 8 fragment rows and columns on.
template <int MT, int WAVES, int CW, class Acc, class Finish>
__device__ __forceinline__ void meet(char* lds, const Acc (&acc)[MT], Finish finish)
{
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    __syncthreads();
    Acc* red = reinterpret_cast<Acc*>(lds);
#pragma unroll
    for (int t = 0; t < MT; ++t)
        red[(wid * MT + t) * 64 + lane] = acc[t];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < MT; ++t)
        if (t == wid)
        {
            Acc v = {0, 0, 0, 0};
            if (CW == 16 || ((lane & 15) < CW && (lane >> 4) < CW / 4))
#pragma unroll
                for (int k = 0; k < WAVES; ++k)
#pragma unroll
                    for (int h = 0; h < 16 / CW; ++h)
                        v += red[(k * MT + t) * 64 + lane + h * 5 * CW];
            finish(t, v);
        }
}

// w: the workgroup's first row of W, ldw bytes apart (16 ldw < 2^32), `rows` of them exist (>= 1; the others repeat the last one and their results are
// not to be stored).  wbytes: bytes of a row of W and of A, a multiple of 16.  xrow(m): row m of A (a valid row also where that one does not
// exist).  At the end wave t calls finish(t, acc), acc[e] = C[16 t + (lane & 15)][first row + 4 (lane >> 4) + e]; with 8 columns only lanes whose
// row and column are below 8 have a result.
template <int WT, class S, class Row, class Finish>
__device__ __forceinline__ void stream(char* lds, const char* w, int64_t ldw, int rows, int wbytes, Row xrow, Finish finish)
{
    using T = Traits<WT>;
    using acc_t = typename T::acc_t;
    static_assert(T::XP == 1, "rows of A as long as W's");
    constexpr int CW = S::cols, WAVES = S::waves, D = S::depth, NX = S::xi, MT = S::mt, STAGE = S::ring / D, NI = NL + NX, BW = CB * 16 / CW;
    static_assert(D <= 2, "the tail's waits");
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); // scalar: M0 and DMA bases
    const int r16 = lane & 15, g4 = lane >> 4, run = r16 / CW;
    char* mine = lds + wid * S::ring;
    const uint32_t ring = (uint32_t) (uintptr_t) (__attribute__((address_space(3))) void*) mine;

    // this lane's piece of request i: fragment row f = 4 i + (lane >> 4), in LDS place lane & 15 of it
    uint32_t woff[NL];
    int wat[NL], xat[NX];
    const char* xr[NX];
#pragma unroll
    for (int i = 0; i < NL; ++i)
    {
        const int f = RPI * i + g4, r = f % CW;
        woff[i] = (uint32_t) ((r < rows ? r : rows - 1) * ldw);
        wat[i] = f / CW * CB + ((r16 ^ f) << 4);
    }
#pragma unroll
    for (int j = 0; j < NX; ++j)
    {
        const int f = RPI * j + g4;
        xr[j] = xrow(CW == 16 ? f : f % CW);
        xat[j] = (CW == 16 ? 0 : f / CW * CB) + ((r16 ^ (f & 15)) << 4);
    }
    const int nblk = (wbytes + BW - 1) / BW;
    const int count = (nblk - wid + WAVES - 1) / WAVES; // blocks wid, wid + WAVES, ...
    auto request = [&](int i) {
        const int base = (wid + i * WAVES) * BW;
        const uint32_t slot = ring + (uint32_t) (i % D) * STAGE;
#pragma unroll
        for (int k = 0; k < NL; ++k)
        {
            const int at = base + wat[k]; // (behind the row: its first piece, dropped below)
            dma_nt(w, woff[k] + (at < wbytes ? at : 0), slot + k * 1024);
        }
#pragma unroll
        for (int j = 0; j < NX; ++j)
        {
            const int at = base + xat[j];
            dma(xr[j] + (at < wbytes ? at : 0), slot + NL * 1024 + j * 1024);
        }
    };

    acc_t acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
        acc[t] = acc_t{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < D; ++i)
        if (i < count)
            request(i);
    for (int i = 0; i < count; ++i)
    {
        if (D > 1 && i + 1 < count)
            wait_requests<(D - 1) * NI>(); // block i is here, the next one under way
        else
            wait_requests<0>();
        const char* st = mine + (i % D) * STAGE;
        const int base = (wid + i * WAVES) * BW;
        const bool whole = base + BW <= wbytes;
#pragma unroll
        for (int s = 0; s < KS; ++s)
        {
            uint4 wf = *reinterpret_cast<const uint4*>(st + r16 * CB + (((s * 4 + g4) ^ r16) << 4));
            uint4 xf[MT];
#pragma unroll
            for (int t = 0; t < MT; ++t)
            {
                const int f = (16 * t + r16) % (RPI * NX);
                xf[t] = *reinterpret_cast<const uint4*>(st + NL * 1024 + f * CB + (((s * 4 + g4) ^ (f & 15)) << 4));
            }
            if (!whole)
            {
                const bool in = base + run * CB + s * 64 + g4 * 16 < wbytes;
                wf = make_uint4(in ? wf.x : 0u, in ? wf.y : 0u, in ? wf.z : 0u, in ? wf.w : 0u);
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    xf[t] = make_uint4(in ? xf[t].x : 0u, in ? xf[t].y : 0u, in ? xf[t].z : 0u, in ? xf[t].w : 0u);
            }
#pragma unroll
            for (int t = 0; t < MT; ++t)
                mma<WT>(acc[t], wf, &xf[t]);
        }
        if (i + D < count)
        {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // the slot has been read
            request(i + D);
        }
    }
    meet<MT, WAVES, CW>(lds, acc, finish);
}

// bytes of LDS of product(): a wave's block of W (the partial sums reuse the room)
template <int MT, int WAVES>
constexpr int lds_bytes()
{
    return WAVES * (16 * CB > MT * 1024 ? 16 * CB : MT * 1024);
}

// As stream(), 16 columns per workgroup.  wbytes: bytes of a W row that hold weights, a multiple of 16.  xrow[t]: this lane's row 16 t + (lane & 15)
// of A (a valid row also where that one does not exist), wbytes * XP bytes.
template <int WT, int MT, int WAVES, class Finish>
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
    uint4 wv[NL], xv[MT][KS * XP];
    auto request = [&](int q) {
        const int base = q * CB;
        const bool w_in = base + lp * 16 < wbytes;
#pragma unroll
        for (int i = 0; i < NL; ++i)
            wv[i] = w_in ? ld_nt16(w + base + woff[i]) : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int s = 0; s < KS; ++s)
        {
            const int at = base + s * 64 + g4 * 16; // of the W row
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int u = 0; u < XP; ++u)
                    xv[t][s * XP + u] = at < wbytes ? *reinterpret_cast<const uint4*>(xrow[t] + (int64_t) at * XP + u * 16) : make_uint4(0, 0, 0, 0);
        }
    };

    acc_t acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
        acc[t] = acc_t{0, 0, 0, 0};

    auto consume = [&]() {
#pragma unroll
        for (int i = 0; i < NL; ++i)
        {
            const int r = RPI * i + lr;
            *reinterpret_cast<uint4*>(mine + r * CB + ((lp ^ (r & 15)) << 4)) = wv[i];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); // (the reads below are of other lanes' pieces)
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int s = 0; s < KS; ++s)
        {
            const uint4 wf = *reinterpret_cast<const uint4*>(mine + r16 * CB + (((s * 4 + g4) ^ r16) << 4));
#pragma unroll
            for (int t = 0; t < MT; ++t)
                mma<WT>(acc[t], wf, &xv[t][s * XP]);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };

    // Blocks wid, wid + WAVES, ...: `count` of them.  In the loop every request is certain - one that might not be made would have the compiler
    // wait as if it had not been.
    const int count = (nblk - wid + WAVES - 1) / WAVES;
    if (count > 0)
    {
        request(wid);
        for (int i = 1; i < count; ++i)
        {
            consume();
            request(wid + i * WAVES);
        }
        consume();
    }
    meet<MT, WAVES, 16>(lds, acc, finish);
}

} // namespace slim
} // namespace dev
} // namespace tllm
