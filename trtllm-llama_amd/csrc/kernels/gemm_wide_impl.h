// Products of many rows on 256 x 256 tiles (those of 128 rows behind them):  C[m,n] = epi( sum_k A[m,k] * W[n,k] ), both operands with K contiguous; bfloat16, fp16 or int8 (the three
// share one geometry: a K-tile is 128 BYTES of every row, a k-step 64 of them, and v_mfma_*_16x16x{32,32,64} takes 16 bytes a lane).  A header, so that
// the translation units that instantiate it for their operand types share one source.  Everything has internal linkage.
//
// What bounds it, and what follows from that (2048 x 4096 x 4096, 128 workgroups, clocks per K-tile of one CU, of which its 512 MFMAs are 2048):
//   * Lock-step stages (barrier, read fragments, multiply) took 3650, the sum of LDS reads and MFMAs: every wave read at the same time.  Here the fragments of
//     the blocks ahead are requested BETWEEN the MFMAs, pinned there, a ring of four A blocks ahead of their use; MFMAs and reads alone 2350.
//   * The operands' way from L2 to LDS alone takes 2260 - 2400 (27 bytes per clock and CU; with 64-byte rows of half as long a K-tile 2900), which is why the tile is the
//     largest that the accumulators allow, rows are whole 128-byte lines, and a K-tile is requested 1.5 K-tiles before its use: A has three buffers, W
//     two, 160 KB together.  W's fragments of a k-step stay in registers, so its buffer is free again halfway through the K-tile: the first of two barriers a
//     K-tile hands over W(t) and A(t - 1) to K-tile t + 2, the second says that K-tile t + 1 has landed.
//   * 16 x 16 MFMAs of twice the depth move half the accumulator traffic of 32 x 32 ones: alone 1.96 against 1.82 PFLOP/s in bfloat16, and where the chip is full
//     its clock falls with its power, 2.2 against 2.0 GHz in the same lock-step kernel.
// All together 2640 - 2700 clocks.  bfloat16, us, in brackets what the lock-step tiles of 32 x 32 MFMAs took: 2048 x 22016 x 4096 gated 285 (350; in a step 315 (353)),
// 4096 x 4096 x 4096 111 (123), 4096 x 8192 x 4096 210 = 1.31 PFLOP/s (265), 1024 x 13056 x 2048 gated 60 (63).
// fp16, in brackets the best of the phased forms of gemm_sqp.hip and of the lock-step ones: 1200 x 12288 x 4096 103 (120), 1200 x 11008 x 4096 95 (112); int8 4096 x 12288 x 4096
// 171 (184), 4096 x 4096 x 4096 59 (67), 4096 x 4096 x 11008 147 = 2.51 POP/s (168).  At 1024 rows, where 256 x 192 tiles fill the chip once, those are quicker (fp16 QKV 87, here 92).
// Tried and slower: the DMA two at a time (+8 %), W's ahead of A's or in turn with them (+10 %), a fifth 64-byte stage, setprio by wave half.
#pragma once
#include "dev_utils.h"
#include "gemm_glds_impl.h"
#include "gemm_seam.h"
#include "kernels.h"
#include "launch_util.h"
#include <algorithm>
#include <cmath>

namespace tllm
{
namespace kernels
{
namespace
{
namespace wide
{
using namespace dev;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void lds_ptr;
typedef const __attribute__((address_space(3))) u32x4* lds_frag;

constexpr int BM = 256, BN = 256, WN = 4, WAVES = 8;
constexpr int NA = 8, NB = 4;               // 16-row blocks of A and of W of a wave (2 x 4 waves)
constexpr int UNIT = 256 * 128;             // bytes of one operand's K-tile
constexpr int LDS_BYTES = 5 * UNIT;         // A: three buffers, W: two
constexpr int AHEAD = 3, RING = 4;          // A blocks requested ahead of their use
constexpr int MID = 5;                      // block of the first k-step in front of which W(t) and A(t - 1) are handed over
constexpr int DMA_A = 4, DMA_W = 4;         // LDS-DMA instructions of a wave and K-tile (8 rows each)

// 64 lanes x 16 bytes, wave-uniform base + a lane's 32-bit offset -> LDS [lds_byte + lane * 16]; in asm, as hipcc would wait for the builtin's in
// front of the next ds_read (it cannot know that it writes another buffer)
__device__ __forceinline__ void load16(const char* base, uint32_t off, uint32_t lds_byte)
{
    uint32_t m0_keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0" : "=&s"(m0_keep) : "v"(off), "s"(base), "s"(lds_byte) : "memory");
}

// LDS image of a K-tile: [row][8 pieces of 16 bytes], piece c of a row at c ^ swz(row).  The lane groups of a ds_read_b128 ({0-3, 12-15, 20-27},
// {4-11, 16-19, 28-31} and + 32) then meet 16 different 16-byte slots.  A lane's row of an A block is lane & 15; of a W block w_row().
__device__ __forceinline__ int a_swz(int row)
{
    return (row & 2) | ((row & 8) >> 1);
}
// Row of W's tile (of the wave's 64) that MFMA row i of block j takes, and with it where a lane's four results of that block go, of row lane & 15.
// PAIRS: blocks 2q and 2q + 1 are together 8 neighbouring columns, 32 q + 8 (lane >> 4) and on: 16 bytes of a 16-bit row; otherwise block j is the 4
// columns 16 j + 4 (lane >> 4) and on: 16 bytes of an fp32 row.  Either way a store covers 64 neighbouring bytes of 16 rows.
template <bool PAIRS>
__device__ __forceinline__ int w_row(int j, int i)
{
    return PAIRS ? 32 * (j >> 1) + 8 * (i >> 2) + 4 * (j & 1) + (i & 3) : 16 * j + i;
}
template <bool PAIRS>
__device__ __forceinline__ int w_swz(int row)
{
    return PAIRS ? (row & 2) | ((row & 16) >> 2) : a_swz(row);
}

template <int WT>
struct Acc
{
    using type = typename std::conditional<WT == W_INT8_SQ, i32x4, f32x4>::type;
};
template <int WT>
__device__ __forceinline__ typename Acc<WT>::type mfma(const u32x4& w, const u32x4& a, const typename Acc<WT>::type& c)
{
    if constexpr (WT == W_INT8_SQ)
        return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, w), __builtin_bit_cast(i32x4, a), c, 0, 0, 0);
    else if constexpr (WT == W_BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, a), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w), __builtin_bit_cast(f16x8, a), c, 0, 0, 0);
}

template <int N>
__device__ __forceinline__ void wait_vm_and_meet()
{
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory");
}

// One wave's part of a tile: its operands' sources and its accumulators.
template <int WT, bool PAIRS>
struct Tile
{
    using acc_t = typename Acc<WT>::type;
    const char *a, *w;      // wave-uniform bases
    uint32_t ao[DMA_A], wo[DMA_W]; // a lane's offsets of its DMA instructions
    uint32_t lds;           // LDS address of the buffers
    int nt, wid, lane;
    acc_t acc[NA][NB];

    __device__ __forceinline__ void dma_a(int i, int t, uint32_t buf) const
    {
        load16(a + (int64_t) t * 128, ao[i], buf + (uint32_t) (i * WAVES + wid) * 1024);
    }
    __device__ __forceinline__ void dma_w(int i, int t, uint32_t buf) const
    {
        load16(w + (int64_t) t * 128, wo[i], buf + (uint32_t) (i * WAVES + wid) * 1024);
    }
    // HALF: the tile has up to 128 rows, the second half of A is not fetched
    template <bool HALF>
    static constexpr int dmas()
    {
        return (HALF ? DMA_A / 2 : DMA_A) + DMA_W;
    }
    // instruction i of K-tile t (A's first, see above)
    template <bool HALF>
    __device__ __forceinline__ void dma(int i, int t, uint32_t abuf, uint32_t wbuf) const
    {
        constexpr int FIRST_W = HALF ? DMA_A / 2 : DMA_A;
        i < FIRST_W ? dma_a(i, t, abuf) : dma_w(i - FIRST_W, t, wbuf);
    }
    // K-tiles 0 and 1
    __device__ __forceinline__ void head(bool half) const
    {
        for (int t = 0; t < 2 && t < nt; ++t)
        {
            const uint32_t ab = lds + (uint32_t) t * UNIT, wb = lds + (uint32_t) (3 + t) * UNIT;
#pragma unroll
            for (int i = 0; i < DMA_A / 2; ++i)
                dma_a(i, t, ab);
            if (!half)
#pragma unroll
                for (int i = DMA_A / 2; i < DMA_A; ++i)
                    dma_a(i, t, ab);
#pragma unroll
            for (int i = 0; i < DMA_W; ++i)
                dma_w(i, t, wb);
        }
    }

    // The K loop, behind a barrier that says that K-tile 0 has landed.  Ends with every wave past its last LDS read.
    template <bool HALF>
    __device__ __forceinline__ void loop()
    {
        uint32_t A0 = lds, A1 = lds + UNIT, A2 = lds + 2 * UNIT, W0 = lds + 3 * UNIT, W1 = lds + 4 * UNIT; // of K-tiles t, t + 1, t + 2 and t, t + 1
        constexpr int DMAS = dmas<HALF>();
        const int wm = wid / WN, wn = wid % WN;
        if (HALF && wm == 1) // no rows: this wave only fetches
        {
            for (int t = 0; t < nt; ++t)
            {
                asm volatile("s_barrier" ::: "memory");
                if (t + 2 < nt)
                {
#pragma unroll
                    for (int i = 0; i < DMAS; ++i)
                        dma<HALF>(i, t + 2, A2, W0);
                    wait_vm_and_meet<DMAS>();
                }
                else
                    wait_vm_and_meet<0>();
                const uint32_t x = A0, y = W0;
                A0 = A1, A1 = A2, A2 = x, W0 = W1, W1 = y;
            }
            asm volatile("s_barrier" ::: "memory");
            return;
        }
        const int i16 = lane & 15, k4 = lane >> 4;
        const uint32_t al = (uint32_t) ((wm * NA * 16 + i16) * 128), wl = (uint32_t) ((wn * NB * 16 + w_row<PAIRS>(0, i16)) * 128);
        const uint32_t as = a_swz(i16), ws = w_swz<PAIRS>(w_row<PAIRS>(0, i16));
        const uint32_t a_k0 = al + ((k4 ^ as) << 4), a_k1 = al + (((4 + k4) ^ as) << 4), w_k0 = wl + ((k4 ^ ws) << 4), w_k1 = wl + (((4 + k4) ^ ws) << 4);
        auto a_at = [](uint32_t base, int block) { return *(lds_frag) (uintptr_t) (base + block * 2048); };
        auto w_at = [](uint32_t base, int j) { return *(lds_frag) (uintptr_t) (base + w_row<PAIRS>(j, 0) * 128); };
        u32x4 fa[RING], fw[2][NB]; // fw: by k-step
#pragma unroll
        for (int j = 0; j < NB; ++j)
            fw[0][j] = w_at(W0 + w_k0, j);
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
            fa[i] = a_at(A0 + a_k0, i);
        for (int t = 0; t < nt; ++t)
        {
            const uint32_t ra0 = A0 + a_k0, ra1 = A0 + a_k1, ran = A1 + a_k0, rw1 = W0 + w_k1, rwn = W1 + w_k0;
            const bool more = t + 2 < nt;
            // every step is pinned (sched_barrier): left to itself the compiler gathers the reads in front of the MFMAs
#pragma unroll
            for (int i = 0; i < NA; ++i) // k-step 0
            {
                if (i == MID)
                {
                    // W's fragments of k-step 1 have arrived (the A blocks requested behind them may still be under way): nobody reads W(t), or A(t - 1), any more
                    asm volatile("s_waitcnt lgkmcnt(%0)\n\ts_barrier" ::"n"(MID - 2) : "memory");
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int j = 0; j < NB; ++j)
                {
                    acc[i][j] = mfma<WT>(fw[0][j], fa[i % RING], acc[i][j]);
                    __builtin_amdgcn_sched_barrier(0);
                    if (j == 0)
                        fa[(i + AHEAD) % RING] = i + AHEAD < NA ? a_at(ra0, i + AHEAD) : a_at(ra1, i + AHEAD - NA);
                    if (i < 2 && (j == 1 || j == 2))
                        fw[1][i * 2 + j - 1] = w_at(rw1, i * 2 + j - 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (i >= MID)
                {
                    if (more && i - MID < DMAS)
                        dma<HALF>(i - MID, t + 2, A2, W0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for (int i = 0; i < NA; ++i) // k-step 1
            {
                if (i == NA - AHEAD)
                {
                    // K-tile t + 1 has landed: this wave's by the count (all of K-tile t + 2's have been requested and stay under way), everyone's by the barrier
                    static_assert(DMAS <= (NA - MID) + (NA - AHEAD), "a K-tile's requests end in front of this wait");
                    if (more)
                        wait_vm_and_meet<DMAS>();
                    else
                        wait_vm_and_meet<0>();
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int j = 0; j < NB; ++j)
                {
                    acc[i][j] = mfma<WT>(fw[1][j], fa[i % RING], acc[i][j]);
                    __builtin_amdgcn_sched_barrier(0);
                    if (j == 0)
                        fa[(i + AHEAD) % RING] = i + AHEAD < NA ? a_at(ra1, i + AHEAD) : a_at(ran, i + AHEAD - NA);
                    const int q = (i - (NA - AHEAD)) * (NB - 1) + j - 1; // (behind the last K-tile: old data, not used)
                    if (i >= NA - AHEAD && j >= 1 && q < NB)
                        fw[0][q] = w_at(rwn, q);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (more && i + NA - MID < DMAS)
                    dma<HALF>(i + NA - MID, t + 2, A2, W0);
                __builtin_amdgcn_sched_barrier(0);
            }
            const uint32_t x = A0, y = W0;
            A0 = A1, A1 = A2, A2 = x, W0 = W1, W1 = y;
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
};

// Where the tiles of a launch are.  Tiles are numbered product by product (or group by group), inside one by bands of eight row tiles, rows fastest; in each round
// of the grid an XCD (workgroups go round them) takes a contiguous range of the numbers, so that the 32 tiles that it works on share 8 + 4 operand panels in its L2.
struct Place
{
    int product, m0, n0, rows, first; // rows: of the product; first: grouped, where they begin
};
__device__ __forceinline__ int rows_to_tiles(int rows)
{
    return (rows + BM - 1) / BM;
}

template <bool GROUPED, int COLS>
struct Places
{
    int tiles_n, total;
    int first, count, own, incl; // grouped, of group `lane` (of 64): where its rows begin, how many, its row tiles, those of all groups up to it

    __device__ __forceinline__ void chunk(const GemmParams& p, int g0, int before, int lane)
    {
        const int g = g0 + lane < p.batch ? g0 + lane : p.batch - 1, lo = p.group_off[g], hi = p.group_off[g + 1];
        first = lo;
        count = hi - lo;
        own = g0 + lane < p.batch ? rows_to_tiles(count) : 0;
        incl = own;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1)
        {
            const int o = __shfl_up(incl, d, 64);
            incl += lane >= d ? o : 0;
        }
        incl += before;
    }
    __device__ __forceinline__ void begin(const GemmParams& p, int lane)
    {
        tiles_n = (p.N + COLS - 1) / COLS;
        if constexpr (!GROUPED)
        {
            total = rows_to_tiles(p.M) * tiles_n * p.batch;
            return;
        }
        int before = 0;
        for (int g0 = 0; g0 < p.batch; g0 += 64)
        {
            chunk(p, g0, before, lane);
            before = __builtin_amdgcn_readlane(incl, 63);
        }
        total = before * tiles_n;
    }
    // the tile of this workgroup's round r; false: there is none left
    __device__ __forceinline__ bool at(const GemmParams& p, int r, int lane, Place& o)
    {
        const int grid = gridDim.x, begin = r * grid, c = blockIdx.x, size = total - begin < grid ? total - begin : grid;
        if (c >= size)
            return false;
        const int q = size >> 3, rest = size & 7, xcd = c & 7;
        int id = begin + (xcd < rest ? xcd * (q + 1) : rest * (q + 1) + (xcd - rest) * q) + (c >> 3);
        o.product = o.first = 0;
        o.rows = p.M;
        if constexpr (GROUPED)
        {
            uint64_t mask;
            for (int g0 = 0, before = 0;; g0 += 64)
            {
                if (p.batch > 64)
                    chunk(p, g0, before, lane); // (else the registers hold the only one)
                o.product = g0;
                mask = __builtin_amdgcn_ballot_w64(id < incl * tiles_n);
                if (mask != 0 || g0 + 64 >= p.batch)
                    break;
                before = __builtin_amdgcn_readlane(incl, 63);
            }
            const int g = mask ? __builtin_ctzll(mask) : 63;
            id -= (__builtin_amdgcn_readlane(incl, g) - __builtin_amdgcn_readlane(own, g)) * tiles_n;
            o.product += g;
            o.first = __builtin_amdgcn_readlane(first, g);
            o.rows = __builtin_amdgcn_readlane(count, g);
        }
        const int tiles_m = rows_to_tiles(o.rows);
        if (!GROUPED && p.batch > 1)
        {
            o.product = id / (tiles_m * tiles_n);
            id -= o.product * (tiles_m * tiles_n);
        }
        constexpr int BAND = 8;
        int band = 0, high = tiles_m;
        if (tiles_m > BAND)
        {
            band = id / (BAND * tiles_n);
            id -= band * (BAND * tiles_n);
            high = tiles_m - band * BAND < BAND ? tiles_m - band * BAND : BAND;
        }
        const int tn = id / high;
        o.m0 = (band * BAND + id - tn * high) * BM;
        o.n0 = tn * COLS;
        return true;
    }
};

// How the results leave: a kernel instance each, as an epilogue's instructions are fetched cold once a tile.
enum Out
{
    OUT_STORE, // c and the output sections: mostly 16-bit rows, bias, relu^2
    OUT_GATED, // gated pairs of columns in front of the first section, 16-bit rows
    OUT_FP32,  // fp32 c alone
    OUT_RESID, // added to the fp32 residual
    OUT_RESID_GATE, // ... behind a sigmoid gate
    OUT_HALF,  // fp16 rows of fp16 or int8 products: scales, fp16 residual or SwiGLU gate
    OUT_DUAL   // two int8 products of the same rows: SwiGLU of both, quantised to int8
};
constexpr bool out_pairs(int out)
{
    return out != OUT_FP32 && out != OUT_RESID && out != OUT_RESID_GATE;
}

__device__ __forceinline__ float4 load4(const float* p)
{
    return *reinterpret_cast<const float4*>(p);
}
__device__ __forceinline__ void store8(float* p, const float (&v)[8])
{
    reinterpret_cast<float4*>(p)[0] = make_float4(v[0], v[1], v[2], v[3]);
    reinterpret_cast<float4*>(p)[1] = make_float4(v[4], v[5], v[6], v[7]);
}
__device__ __forceinline__ uint32_t bf_pair(float a, float b)
{
    return (uint32_t) f2bf(a) | ((uint32_t) f2bf(b) << 16);
}
__device__ __forceinline__ void store8(uint16_t* p, const float (&v)[8])
{
    *reinterpret_cast<uint4*>(p) = make_uint4(bf_pair(v[0], v[1]), bf_pair(v[2], v[3]), bf_pair(v[4], v[5]), bf_pair(v[6], v[7]));
}

// bfloat16 products: the stack engine's layer seam.  Offsets and addresses are whole 16-byte pieces, fp32 sections without an activation apart (serves()); c: of this product
template <int OUT, int NA, int NB>
__device__ __forceinline__ void leave_pairs(const GemmParams& p, const f32x4 (&acc)[NA][NB], int lane, void* c, int row0, int col0, int rows)
{
#pragma unroll
    for (int jp = 0; jp < NB / 2; ++jp)
    {
        const int col = col0 + 32 * jp + 8 * (lane >> 4);
        if (col >= p.N)
            continue;
        float b[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (p.bias)
        {
            const float4 x = load4(p.bias + col), y = load4(p.bias + col + 4);
            b[0] = x.x, b[1] = x.y, b[2] = x.z, b[3] = x.w, b[4] = y.x, b[5] = y.y, b[6] = y.z, b[7] = y.w;
        }
        const SeamOut so = seam_out<false>(p.seam, p.act, c, p.ldc, p.out_dtype != DT_BFLOAT16, col);
        auto value = [&](float (&v)[8], int i) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                v[e] = acc[i][2 * jp + (e >> 2)][e & 3] + b[e];
        };
        auto rows_out = [&](auto* to) {
#pragma unroll
            for (int i = 0; i < NA; ++i)
            {
                float v[8];
                value(v, i);
                if (so.act == GEMM_ACT_RELU2)
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        v[e] = seam_relu2(v[e]);
                if (row0 + i * 16 < rows)
                    store8(to + (int64_t) (row0 + i * 16) * so.ldc + col, v);
            }
        };
        if (OUT == OUT_GATED && seam_gated(so.act))
        {
#pragma unroll
            for (int i = 0; i < NA; ++i)
            {
                float v[8], g[4];
                value(v, i);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    g[e] = seam_gate<false>(p.act, v[2 * e], v[2 * e + 1]);
                if (row0 + i * 16 < rows)
                    *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(so.c) + (int64_t) (row0 + i * 16) * so.ldc + (col >> 1)) = make_uint2(bf_pair(g[0], g[1]), bf_pair(g[2], g[3]));
            }
        }
        else if (so.f32)
        {
            float* to = reinterpret_cast<float*>(so.c);
            if (col + 8 <= p.N && !((reinterpret_cast<uintptr_t>(to + col) | (so.ldc << 2)) & 15))
                rows_out(to);
            else // a section of a few columns
#pragma unroll
                for (int i = 0; i < NA; ++i)
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (col + e < p.N && row0 + i * 16 < rows)
                            to[(int64_t) (row0 + i * 16) * so.ldc + col + e] = acc[i][2 * jp + (e >> 2)][e & 3] + b[e];
        }
        else
            rows_out(reinterpret_cast<uint16_t*>(so.c));
    }
}
template <int OUT, int NA, int NB>
__device__ __forceinline__ void leave_fp32(const GemmParams& p, const f32x4 (&acc)[NA][NB], int lane, void* c, int row0, int col0, int rows)
{
#pragma clang fp contract(off) // (the gated product is rounded before it is added, as gemm_glds_impl.h leaves it)
    float* out = OUT == OUT_FP32 ? reinterpret_cast<float*>(c) : p.resid;
    const int64_t ld = OUT == OUT_FP32 ? p.ldc : p.ldr;
#pragma unroll
    for (int j = 0; j < NB; ++j)
    {
        const int col = col0 + 16 * j + 4 * (lane >> 4);
        if (col >= p.N)
            continue;
        const float* bias = OUT == OUT_RESID_GATE ? p.gate_bias : p.bias;
        float4 b = make_float4(0.f, 0.f, 0.f, 0.f);
        if (OUT != OUT_RESID && bias)
            b = load4(bias + col);
#pragma unroll
        for (int i = 0; i < NA; ++i)
        {
            const int64_t row = row0 + i * 16;
            if (row >= rows)
                continue;
            float* at = out + row * ld + col;
            float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
            if constexpr (OUT == OUT_FP32)
                *reinterpret_cast<float4*>(at) = make_float4(v[0] + b.x, v[1] + b.y, v[2] + b.z, v[3] + b.w);
            else
            {
                const float4 o = load4(at);
                if constexpr (OUT == OUT_RESID_GATE)
                {
                    const uint2 z = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(p.gate) + row * p.ldg + col);
                    v[0] *= 1.f / (1.f + __expf(-(__builtin_bit_cast(float, z.x << 16) + b.x)));
                    v[1] *= 1.f / (1.f + __expf(-(__builtin_bit_cast(float, z.x & 0xffff0000u) + b.y)));
                    v[2] *= 1.f / (1.f + __expf(-(__builtin_bit_cast(float, z.y << 16) + b.z)));
                    v[3] *= 1.f / (1.f + __expf(-(__builtin_bit_cast(float, z.y & 0xffff0000u) + b.w)));
                }
                *reinterpret_cast<float4*>(at) = make_float4(o.x + v[0], o.y + v[1], o.z + v[2], o.w + v[3]);
            }
        }
    }
}

// fp16 and int8 products: the scales of a lane's columns and rows, requested ahead of the K loop (behind it they would wait for the next tile's first requests)
template <int WT, int OUT, int NA = wide::NA, int NB = wide::NB>
struct Scales
{
    // int8: factors of the columns of block pair q (OUT_DUAL: of the first and the second product) and of the rows; fp16: weight-only's of a column
    float col[NB / 2][8], row[WT == W_INT8_SQ && OUT == OUT_HALF ? NA : 1];

    __device__ __forceinline__ void request(const GemmParams& p, int row0, int col0, int rows, int lane)
    {
#pragma unroll
        for (int q = 0; q < NB / 2; ++q)
        {
            int c = col0 + (OUT == OUT_DUAL ? 0 : 32 * q) + 8 * (lane >> 4);
            c = c < p.N ? c : 0;
            if constexpr (WT == W_INT8_SQ)
            {
                const float* from = reinterpret_cast<const float*>(OUT == OUT_DUAL && q ? p.scale_col2 : p.scale_col);
                if (p.per_channel)
                {
                    const float4 x = load4(from + c), y = load4(from + c + 4);
                    col[q][0] = x.x, col[q][1] = x.y, col[q][2] = x.z, col[q][3] = x.w, col[q][4] = y.x, col[q][5] = y.y, col[q][6] = y.z, col[q][7] = y.w;
                }
                else
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        col[q][e] = from[0];
            }
            else
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    col[q][e] = p.scale_col ? h2f(reinterpret_cast<const uint16_t*>(p.scale_col)[c + e]) : 1.f;
        }
        if constexpr (WT == W_INT8_SQ)
#pragma unroll
            for (int i = 0; i < (int) (sizeof(row) / sizeof(row[0])); ++i)
            {
                const int m = row0 + i * 16;
                row[i] = p.scale_row[OUT == OUT_HALF && p.per_token ? (m < rows ? m : rows - 1) : 0];
            }
    }
};
__device__ __forceinline__ uint32_t half_pair(float a, float b)
{
    return (uint32_t) f2h(a) | ((uint32_t) f2h(b) << 16);
}
template <int WT, int NA, int NB>
__device__ __forceinline__ void leave_half(const GemmParams& p, const typename Acc<WT>::type (&acc)[NA][NB], int lane, const Scales<WT, OUT_HALF, NA, NB>& sc, int row0, int col0, int rows)
{
    auto out = [&](auto finish) {
#pragma unroll
        for (int q = 0; q < NB / 2; ++q)
        {
            const int col = col0 + 32 * q + 8 * (lane >> 4);
            if (col >= p.N)
                continue;
#pragma unroll
            for (int i = 0; i < NA; ++i)
            {
                if (row0 + i * 16 >= rows)
                    continue;
                float v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e)
                {
                    const auto a = acc[i][2 * q + (e >> 2)][e & 3];
                    if constexpr (WT == W_INT8_SQ)
                        v[e] = (float) a * (sc.col[q][e] * sc.row[i]);
                    else
                        v[e] = a * sc.col[q][e];
                }
                const int64_t at = (int64_t) (row0 + i * 16) * p.ldc + col;
                *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(p.c) + at)
                    = finish(make_uint4(half_pair(v[0], v[1]), half_pair(v[2], v[3]), half_pair(v[4], v[5]), half_pair(v[6], v[7])), at);
            }
        }
    };
    if (p.residual)
        out([&](const uint4& v, int64_t at) {
            const uint4 r = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(p.residual) + at);
            const uint32_t a[4] = {v.x, v.y, v.z, v.w}, b[4] = {r.x, r.y, r.z, r.w};
            uint32_t o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                o[e] = half_pair(h2f((uint16_t) (a[e] & 0xffffu)) + h2f((uint16_t) (b[e] & 0xffffu)), h2f((uint16_t) (a[e] >> 16)) + h2f((uint16_t) (b[e] >> 16)));
            return make_uint4(o[0], o[1], o[2], o[3]);
        });
    else if (WT == W_FP16 && p.silu_gate)
        out([&](const uint4& v, int64_t at) { return epi_silu_gate8(v, *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(p.silu_gate) + at)); });
    else
        out([](const uint4& v, int64_t) { return v; });
}
// rounded where two fp16 products, SwiGLU in fp16 and the static quantiser would round
__device__ __forceinline__ void leave_dual(const GemmParams& p, const Tile<W_INT8_SQ, true>& t, const Scales<W_INT8_SQ, OUT_DUAL>& sc, int row0, int col0, int rows)
{
    const int col = col0 + 8 * (t.lane >> 4);
    if (col >= p.N)
        return;
    const float qs = p.swiglu_qscale[0], sr2 = p.scale_row2 ? p.scale_row2[0] : p.scale_row[0];
#pragma unroll
    for (int i = 0; i < NA; ++i)
    {
        uint32_t o[2] = {0, 0};
#pragma unroll
        for (int e = 0; e < 8; ++e)
        {
            const float g16 = h2f(f2h((float) t.acc[i][e >> 2][e & 3] * (sc.col[0][e] * sc.row[0])));
            const float u16 = h2f(f2h((float) t.acc[i][2 + (e >> 2)][e & 3] * (sc.col[1][e] * sr2)));
            const float a16 = h2f(f2h(g16 / (1.f + __expf(-g16))));
            const float o16 = h2f(f2h(a16 * u16));
            o[e >> 2] |= ((uint32_t) (uint8_t) f2i8_rni_sat(o16 * qs)) << (8 * (e & 3));
        }
        if (row0 + i * 16 < rows)
            *reinterpret_cast<uint2*>(reinterpret_cast<int8_t*>(p.c) + (int64_t) (row0 + i * 16) * p.ldc + col) = make_uint2(o[0], o[1]);
    }
}

// Persistent: a workgroup per CU (fewer where that makes the rounds even) walks its tiles; the next tile's first two K-tiles are under way while this
// one's results leave, straight from the accumulators (16 rows x 64 bytes a store, no LDS).  The code in front of the first request runs cold: one copy
// of it serves the first tile and the others (2.2 us with two, a batch's and a group's places in one instance and K-tile 1's requests unrolled).
template <int WT, int OUT, bool GROUPED>
__global__ __launch_bounds__(64 * WAVES) void wide_kernel(const GemmParams p)
{
    extern __shared__ __attribute__((aligned(16))) char wide_lds[];
    constexpr int ES = WT == W_INT8_SQ ? 1 : 2;
    constexpr bool PAIRS = out_pairs(OUT);
    using T = Tile<WT, PAIRS>;
    T t;
    t.lane = threadIdx.x & 63;
    t.wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    t.lds = (uint32_t) (uintptr_t) (lds_ptr*) wide_lds;
    t.nt = p.K * ES / 128;
    constexpr bool DUAL = OUT == OUT_DUAL;
    Places<GROUPED, DUAL ? BN / 2 : BN> places;
    places.begin(p, t.lane);
    Place now = {}, next;
    Scales<WT, OUT> scales;
    for (int round = 0;; ++round)
    {
        const bool more = places.at(p, round, t.lane, next);
        const bool half = next.rows - next.m0 <= BM / 2;
        if (more)
        {
            const int row8 = t.wid * 8 + (t.lane >> 3), piece = t.lane & 7;
            t.a = reinterpret_cast<const char*>(p.a);
            t.w = reinterpret_cast<const char*>(DUAL && t.wid >= WAVES / 2 ? p.w2 : p.w);
            if (WT == W_BF16 && (GROUPED || p.batch > 1))
            {
                t.a += GROUPED ? 0 : next.product * p.batch_a;
                t.w += next.product * p.batch_w;
            }
#pragma unroll
            for (int i = 0; i < DMA_A; ++i)
            {
                const int row = i * WAVES * 8 + row8, m = next.m0 + row;
                int r = next.first + (m < next.rows ? m : next.rows - 1);
                if (GROUPED && p.a_rows)
                    r = p.a_rows[r];
                t.ao[i] = (uint32_t) r * (uint32_t) (p.lda * ES) + ((piece ^ a_swz(row)) << 4);
            }
#pragma unroll
            for (int i = 0; i < DMA_W; ++i)
            {
                // two products: the first 32 of a wave's 64 rows are the first matrix's, the others the second one's
                const int row = i * WAVES * 8 + row8, col = next.n0 + (DUAL ? 32 * i + (row8 & 31) : row), n = col < p.N ? col : p.N - 1;
                t.wo[i] = (uint32_t) n * (uint32_t) p.ldw + ((piece ^ w_swz<PAIRS>(row)) << 4);
            }
            t.head(half);
        }
        const int row0 = now.m0 + t.wid / WN * (NA * 16) + (t.lane & 15), col0 = now.n0 + t.wid % WN * (DUAL ? NB * 8 : NB * 16);
        if (round > 0)
        {
            if constexpr (WT == W_BF16)
            {
                char* c = reinterpret_cast<char*>(p.c);
                c += GROUPED ? now.first * p.ldc * (p.out_dtype == DT_FLOAT ? 4 : 2) : now.product * p.batch_c;
                if constexpr (PAIRS)
                    leave_pairs<OUT>(p, t.acc, t.lane, c, row0, col0, now.rows);
                else
                    leave_fp32<OUT>(p, t.acc, t.lane, c, row0, col0, now.rows);
            }
            else if constexpr (DUAL)
                leave_dual(p, t, scales, row0, col0, now.rows);
            else
                leave_half<WT, NA, NB>(p, t.acc, t.lane, scales, row0, col0, now.rows);
        }
        if (!more)
            return;
        now = next;
        if (round == 0 && t.nt > 1)
        {
            if (half)
                wait_vm_and_meet<T::template dmas<true>()>();
            else
                wait_vm_and_meet<T::template dmas<false>()>();
        }
        else
            wait_vm_and_meet<0>(); // (the results of the tile before have left, too)
        if constexpr (WT != W_BF16)
            scales.request(p, now.m0 + t.wid / WN * (NA * 16) + (t.lane & 15), now.n0 + t.wid % WN * (DUAL ? NB * 8 : NB * 16), now.rows, t.lane);
#pragma unroll
        for (int i = 0; i < NA; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
                t.acc[i][j] = typename T::acc_t{0, 0, 0, 0};
        if (half)
            t.template loop<true>();
        else
            t.template loop<false>();
    }
}

// Tiles of 128 rows, for products of few tiles and groups of few rows: a tile a workgroup of 8 waves, S whole stages of 128-byte rows, results straight from the
// accumulators as above.  PINNED: reads between the MFMAs, one barrier a K-tile (128 x 256 and 128 x 192); otherwise a k-step's reads in front of its MFMAs, which
// the SIMD's other wave covers (128 x 128 and 128 x 64: pinned reads gave them nothing).  Bound by the operands' way from L2 and, once a wave's MFMAs are queued, by
// them: 128 x 256 1600 - 1800 clocks a K-tile, 1024 of them MFMAs.  us in a step, in brackets the lock-step tiles of 32 x 32 MFMAs whose results went through LDS:
//   128 x 256  2048 x 4096 x 4096 65 (70), x 11008 168 (180), 1672 x 4096 x 2048 35 (41), 32 groups of 8192 rows, 5504, 4096 493 (514), of 6688 rows, 2816, 2048 127 (126)
//   128 x 192  1024 x 6912 x 2048 29.5 (31.9), 2048 x 8832 x 4096 161 (165)      128 x 128  1672 x 2048 x 2048 14.5 (17.8)
//   128 x 64   1024 x 2048 x 4096 and x 6528, behind a gate into the residual 29.8 (31.7)
//   (fp16 and int8, whole fp16 pieces: figures at the rule that picks them, gemm_glds.hip)
// (Named as the lock-step form: whoever reads a tile from a kernel's name finds it in the same arguments; wide:: tells the two apart.)
template <int WT, int WM, int WN, int MT, int NT, int S, int OUT, bool GROUPED, bool PINNED>
__global__ __launch_bounds__(64 * WM * WN) void gemm_glds_kernel(const GemmParams p_in)
{
    static_assert(WT == W_BF16 || (OUT == OUT_HALF && !GROUPED), "what the other two types leave");
    constexpr bool PAIRS = out_pairs(OUT);
    constexpr int ES = WT == W_INT8_SQ ? 1 : 2, NA = 2 * MT, NB = 2 * NT;
    constexpr int NW = WM * WN, BM = WM * NA * 16, BN = WN * NB * 16, STAGE = (BM + BN) * 128, DMAS = (BM + BN) / 8 / NW, DMA_A = BM / 8 / NW;
    static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "whole instructions");
    extern __shared__ __attribute__((aligned(16))) char wide_lds[];
    GemmParams p = p_in;
    const bool clocked = WT == W_INT8_SQ && p.clock_probe; // (microbench hook)
    const uint64_t clk0 = clocked ? __builtin_readcyclecounter() : 0, rt0 = clocked ? __builtin_amdgcn_s_memrealtime() : 0;
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wid / WN, wn = wid % WN;
    int64_t product = blockIdx.y;
    int id = blockIdx.x;
    if constexpr (GROUPED)
    {
        const GroupTile gt = group_tile<BM>(p, (p.N + BN - 1) / BN, id);
        if (gt.group < 0)
            return; // behind the last tile
        product = gt.group;
        id = gt.tile;
        const int64_t o = p.group_off[product];
        p.M = p.group_off[product + 1] - (int) o;
        if (p.a_rows)
            p.a_rows += o;
        else
            p.a = reinterpret_cast<const char*>(p.a) + o * p.lda * 2;
        p.c = reinterpret_cast<char*>(p.c) + o * p.ldc * (p.out_dtype == DT_FLOAT ? 4 : 2);
    }
    else
    {
        // each XCD a contiguous range of the tiles, row tiles fastest: those that share a panel of W run side by side on one L2
        const int q = gridDim.x >> 3, r = gridDim.x & 7, xcd = id & 7;
        id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (id >> 3);
        if constexpr (WT == W_BF16)
        {
            p.a = reinterpret_cast<const char*>(p.a) + product * p.batch_a;
            p.c = reinterpret_cast<char*>(p.c) + product * p.batch_c;
        }
    }
    const char* w = reinterpret_cast<const char*>(p.w) + (WT == W_BF16 ? product * p.batch_w : 0);
    const int tiles_m = (p.M + BM - 1) / BM, tn = id / tiles_m, m0 = (id - tn * tiles_m) * BM, n0 = tn * BN, nt = p.K * ES / 128;
    const uint32_t lds = (uint32_t) (uintptr_t) (lds_ptr*) wide_lds;
    uint32_t from[DMAS];
#pragma unroll
    for (int i = 0; i < DMAS; ++i)
    {
        const int row = ((i < DMA_A ? i : i - DMA_A) * NW + wid) * 8 + (lane >> 3);
        if (i < DMA_A)
        {
            int r = m0 + row < p.M ? m0 + row : p.M - 1;
            if (GROUPED && p.a_rows)
                r = p.a_rows[r];
            from[i] = (uint32_t) r * (uint32_t) (p.lda * ES) + (((lane & 7) ^ a_swz(row)) << 4);
        }
        else
            from[i] = (uint32_t) (n0 + row < p.N ? n0 + row : p.N - 1) * (uint32_t) p.ldw + (((lane & 7) ^ w_swz<PAIRS>(row)) << 4);
    }
    auto dma = [&](int i, int t, uint32_t stage) {
        load16((i < DMA_A ? reinterpret_cast<const char*>(p.a) : w) + (int64_t) t * 128, from[i], stage + (uint32_t) (i * NW + wid) * 1024);
    };
    using acc_t = typename Acc<WT>::type;
    acc_t acc[NA][NB];
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
            acc[i][j] = acc_t{0, 0, 0, 0};
    const int i16 = lane & 15, k4 = lane >> 4;
    const uint32_t al = (uint32_t) ((wm * NA * 16 + i16) * 128), wl = (uint32_t) (BM * 128 + (wn * NB * 16 + w_row<PAIRS>(0, i16)) * 128);
    const uint32_t as = a_swz(i16), ws = w_swz<PAIRS>(w_row<PAIRS>(0, i16));
    const uint32_t a_k[2] = {al + ((k4 ^ as) << 4), al + (((4 + k4) ^ as) << 4)}, w_k[2] = {wl + ((k4 ^ ws) << 4), wl + (((4 + k4) ^ ws) << 4)};
    auto a_at = [](uint32_t base, int block) { return *(lds_frag) (uintptr_t) (base + block * 2048); };
    auto w_at = [](uint32_t base, int j) { return *(lds_frag) (uintptr_t) (base + w_row<PAIRS>(j, 0) * 128); };
    const uint32_t end = lds + S * STAGE;
    const int row0 = m0 + wm * (NA * 16) + i16, col0 = n0 + wn * (NB * 16);
    Scales<WT, OUT, NA, NB> scales;
    if constexpr (WT != W_BF16)
        scales.request(p, row0, col0, p.M, lane);
    if constexpr (PINNED)
    {
        constexpr int BLOCKS = 2 * NA, L = BLOCKS >= 8 ? 3 : 2, HAND_OVER = BLOCKS - L;
#pragma unroll
        for (int t = 0; t < S; ++t)
            if (t < nt)
#pragma unroll
                for (int i = 0; i < DMAS; ++i)
                    dma(i, t, lds + t * STAGE);
        if (nt >= S)
            wait_vm_and_meet<(S - 1) * DMAS>();
        else
            wait_vm_and_meet<0>();
        u32x4 fa[BLOCKS + L], fw[2][NB]; // fa: by block, those of the next stage behind; renamed, not kept
#pragma unroll
        for (int j = 0; j < NB; ++j)
            fw[0][j] = w_at(lds + w_k[0], j);
#pragma unroll
        for (int i = 0; i < L; ++i)
            fa[i] = a_at(lds + a_k[0], i);
        uint32_t cur = lds, before = lds;
        for (int t = 0; t < nt; ++t)
        {
            const uint32_t next = cur + STAGE == end ? lds : cur + STAGE;
            const uint32_t ra[3] = {cur + a_k[0], cur + a_k[1], next + a_k[0]}, rw1 = cur + w_k[1], rwn = next + w_k[0];
#pragma unroll
            for (int g = 0; g < BLOCKS; ++g)
            {
                if (g == HAND_OVER)
                {
                    // stage t + 1 has landed, nobody reads stage t any more: its room is for stage t + S
                    if (t + S - 1 < nt)
                        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((S - 2) * DMAS) : "memory");
                    else
                        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int j = 0; j < NB; ++j)
                {
                    acc[g % NA][j] = mfma<WT>(fw[g / NA][j], fa[g], acc[g % NA][j]);
                    __builtin_amdgcn_sched_barrier(0);
                    if (j == 0)
                        fa[g + L] = a_at(ra[(g + L) / NA], (g + L) % NA);
                    else
                    {
                        const int q = g * (NB - 1) + j - 1, qn = q - HAND_OVER * (NB - 1);
                        if (q < NB)
                            fw[1][q] = w_at(rw1, q);
                        if (qn >= 0 && qn < NB) // (behind the last stage: old data, not used)
                            fw[0][qn] = w_at(rwn, qn);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                // stage t - 1 + S, into the room that the hand-over from t - 1 to t released
#pragma unroll
                for (int i = 0; i < DMAS; ++i)
                    if (g < HAND_OVER && i * HAND_OVER / DMAS == g)
                    {
                        if (t >= 1 && t - 1 + S < nt)
                            dma(i, t - 1 + S, before);
                        __builtin_amdgcn_sched_barrier(0);
                    }
            }
#pragma unroll
            for (int i = 0; i < L; ++i)
                fa[i] = fa[BLOCKS + i];
            before = cur;
            cur = next;
        }
    }
    else
    {
        constexpr int AHEAD_STAGES = S - 1, PARTS = 2;
#pragma unroll
        for (int t = 0; t < AHEAD_STAGES; ++t)
            if (t < nt)
#pragma unroll
                for (int i = 0; i < DMAS; ++i)
                    dma(i, t, lds + t * STAGE);
        uint32_t cur = lds, into = lds + AHEAD_STAGES * STAGE;
        for (int t = 0; t < nt; ++t)
        {
            // stage t has landed (the younger ones stay under way), and nobody reads stage t - 1 any more, whose room the next requests take
            if (t + AHEAD_STAGES - 1 < nt)
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((AHEAD_STAGES - 1) * DMAS) : "memory");
            else
                asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
            for (int k = 0; k < 2; ++k)
            {
                u32x4 fa[NA], fw[NB];
#pragma unroll
                for (int i = 0; i < NA; ++i)
                    fa[i] = a_at(cur + a_k[k], i);
#pragma unroll
                for (int j = 0; j < NB; ++j)
                    fw[j] = w_at(cur + w_k[k], j);
                __builtin_amdgcn_sched_barrier(0);
                if (t + AHEAD_STAGES < nt)
#pragma unroll
                    for (int i = 0; i < DMAS; ++i)
                        if (i % PARTS == k)
                            dma(i, t + AHEAD_STAGES, into);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < NA; ++i)
#pragma unroll
                    for (int j = 0; j < NB; ++j)
                        acc[i][j] = mfma<WT>(fw[j], fa[i], acc[i][j]);
            }
            cur = cur + STAGE == end ? lds : cur + STAGE;
            into = into + STAGE == end ? lds : into + STAGE;
        }
    }
    if constexpr (WT != W_BF16)
    {
        leave_half<WT, NA, NB>(p, acc, lane, scales, row0, col0, p.M);
        if (clocked && threadIdx.x == 0)
        {
            uint64_t* to = reinterpret_cast<uint64_t*>(p.clock_probe) + 2 * blockIdx.x;
            to[0] = __builtin_readcyclecounter() - clk0;
            to[1] = __builtin_amdgcn_s_memrealtime() - rt0;
        }
    }
    else if constexpr (PAIRS)
        leave_pairs<OUT>(p, acc, lane, p.c, row0, col0, p.M);
    else
        leave_fp32<OUT>(p, acc, lane, p.c, row0, col0, p.M);
}

// Tiles of up to 288 rows x 192 columns, for groups of a few hundred rows: bfloat16, 8 waves of 2 x 4, a wave the row blocks wm, wm + 2, ... and 48 columns.  A group's rows
// are cut into as few tiles as take them, of equal height in steps of 32 rows; a wave's blocks are a template of the loop, so that a tile fetches and multiplies no more rows than it has
// (but for tiles of up to 64 rows, which go by the loop of 96).
//   Bound by the operands' way from L2 (28 bytes per clock and CU) and the weights' from HBM.  Tiles of 128 rows bring a group's weights in two or three times, the last one for
// a few rows as often as not; 256 x 256 ones once, but a group of a few rows more costs two thirds of another tile, and a tile is a third of a round: that is why a tile is
// as high as three buffers of A and two of W's 192 columns let it be.  Reads and requests as in the 256 x 256 loop: 1.5 K-tiles ahead, W's buffer handed back within the K-tile.
// us, 32 groups, random sizes, cold weights, in brackets 128 x 256 and 256 x 256: 8192 rows, 5504, 4096 390 (476, 523; 330 with weights from L2), 4096, 2752 216 (272, 295), 6900 rows,
// 2816, 2048 111 (122, 130; 84 with weights from L2), of 12000 rows, 4224, 3072 338 (392, 400).
// Tried and no quicker: W asked for two K-tiles ahead and A three where they fit (nothing: it is not the latency), weights' requests marked nt, K begun at another place by each column of
// tiles (100 -> 87 at 4084 rows, 2816, 2048, whose rows of 4096 bytes meet few memory channels, 390 -> 460 at 5504, 4096).
template <int NA>
struct TallLoop
{
    static constexpr int NB = 3, BLOCKS = 2 * NA, AHEAD = NA >= 5 ? 3 : 2, HAND_OVER = BLOCKS - AHEAD, MID = NA >= 5 ? 3 : 2;
    static constexpr int DMA_A = (NA + 1) / 2, DMA_W = 3, DMAS = DMA_A + DMA_W, SLOTS = (HAND_OVER - MID) * NB;
    static constexpr bool ODD = NA % 2 != 0; // the last of A's requests is there in half of the waves only
};
constexpr int TALL_BM = 288, TALL_BN = 192, TALL_A = TALL_BM * 128, TALL_W = TALL_BN * 128, TALL_LDS = 3 * TALL_A + 2 * TALL_W;
// Row of W's tile (of the wave's 48) that MFMA row i of block j takes: a lane's results of the three blocks are 12 neighbouring columns.
__device__ __forceinline__ int tall_w_row(int j, int i)
{
    return 12 * (i >> 2) + 4 * j + (i & 3);
}
__device__ __forceinline__ int tall_w_swz(int row) // of 192
{
    return (row & 2) | (row % 48 >= 24 ? 4 : 0);
}
struct TallTile
{
    const char *a, *w;
    uint32_t ao[5], wo[3], lds;
    int nt, wid, lane;
    f32x4 acc[9][3];

    template <int NA>
    __device__ __forceinline__ void dma(int i, int t, uint32_t abuf, uint32_t wbuf) const
    {
        using L = TallLoop<NA>;
        if (i >= L::DMA_A)
            load16(w + (int64_t) t * 128, wo[i - L::DMA_A], wbuf + (uint32_t) ((i - L::DMA_A) * 8 + wid) * 1024);
        else if (!L::ODD || i < L::DMA_A - 1 || wid < 4)
            load16(a + (int64_t) t * 128, ao[i], abuf + (uint32_t) (i * 8 + wid) * 1024);
    }
    // this wave's requests are in but for the last K-tile's, everyone's behind the barrier
    template <int NA>
    __device__ __forceinline__ void landed() const
    {
        using L = TallLoop<NA>;
        if (L::ODD && wid >= 4)
            wait_vm_and_meet<L::DMAS - 1>();
        else
            wait_vm_and_meet<L::DMAS>();
    }
    template <int NA>
    __device__ __forceinline__ void run()
    {
        using L = TallLoop<NA>;
        constexpr int NB = L::NB;
        static_assert(L::SLOTS > 0 && L::AHEAD * (NB - 1) >= NB, "requests between the two barriers, the next k-step's fragments behind the second");
        uint32_t A0 = lds, A1 = lds + TALL_A, A2 = lds + 2 * TALL_A, W0 = lds + 3 * TALL_A, W1 = W0 + TALL_W; // of K-tiles t, t + 1, t + 2 and t, t + 1
#pragma unroll
        for (int i = 0; i < L::DMAS; ++i)
            dma<NA>(i, 0, A0, W0);
#pragma unroll
        for (int i = 0; i < L::DMAS; ++i)
            dma<NA>(i, 1, A1, W1);
        landed<NA>();
#pragma unroll
        for (int i = 0; i < NA; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
                acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int i16 = lane & 15, k4 = lane >> 4, wm = wid >> 2, wn = wid & 3;
        const uint32_t al = (uint32_t) ((16 * wm + i16) * 128), wl = (uint32_t) ((48 * wn + tall_w_row(0, i16)) * 128);
        const uint32_t as = a_swz(i16), ws = tall_w_swz(tall_w_row(0, i16));
        const uint32_t a_k0 = al + ((k4 ^ as) << 4), a_k1 = al + (((4 + k4) ^ as) << 4), w_k0 = wl + ((k4 ^ ws) << 4), w_k1 = wl + (((4 + k4) ^ ws) << 4);
        auto a_at = [](uint32_t base, int block) { return *(lds_frag) (uintptr_t) (base + block * 4096); };
        auto w_at = [](uint32_t base, int j) { return *(lds_frag) (uintptr_t) (base + j * 512); };
        u32x4 fa[L::BLOCKS + L::AHEAD], fw[2][NB];
#pragma unroll
        for (int j = 0; j < NB; ++j)
            fw[0][j] = w_at(W0 + w_k0, j);
#pragma unroll
        for (int i = 0; i < L::AHEAD; ++i)
            fa[i] = a_at(A0 + a_k0, i);
        for (int t = 0; t < nt; ++t)
        {
            const uint32_t ra[3] = {A0 + a_k0, A0 + a_k1, A1 + a_k0}, rw1 = W0 + w_k1, rwn = W1 + w_k0;
            const bool more = t + 2 < nt;
#pragma unroll
            for (int g = 0; g < L::BLOCKS; ++g)
            {
                if (g == L::MID)
                {
                    // W's fragments of k-step 1 have arrived (A blocks requested behind them may be under way): nobody reads W(t), or A(t - 1), any more
                    asm volatile("s_waitcnt lgkmcnt(%0)\n\ts_barrier" ::"n"(L::MID - 2) : "memory");
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (g == L::HAND_OVER)
                {
                    // K-tile t + 1 has landed
                    if (more)
                        landed<NA>();
                    else
                        wait_vm_and_meet<0>();
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int j = 0; j < NB; ++j)
                {
                    acc[g % NA][j] = mfma<W_BF16>(fw[g / NA][j], fa[g], acc[g % NA][j]);
                    __builtin_amdgcn_sched_barrier(0);
                    if (j == 0)
                        fa[g + L::AHEAD] = a_at(ra[(g + L::AHEAD) / NA], (g + L::AHEAD) % NA);
                    else
                    {
                        const int q = g * (NB - 1) + j - 1, qn = q - L::HAND_OVER * (NB - 1);
                        if (q < NB)
                            fw[1][q] = w_at(rw1, q);
                        if (qn >= 0 && qn < NB) // (behind the last K-tile: old data, not used)
                            fw[0][qn] = w_at(rwn, qn);
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int i = 0; i < L::DMAS; ++i)
                        if (more && g >= L::MID && g < L::HAND_OVER && i * L::SLOTS / L::DMAS == (g - L::MID) * NB + j)
                            dma<NA>(i, t + 2, A2, W0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for (int i = 0; i < L::AHEAD; ++i)
                fa[i] = fa[L::BLOCKS + i];
            const uint32_t x = A0, y = W0;
            A0 = A1, A1 = A2, A2 = x, W0 = W1, W1 = y;
        }
    }
    template <int OUT, int NA>
    __device__ __forceinline__ void leave(const GemmParams& p, char* c, int row0, int col, int rows) const
    {
#pragma unroll
        for (int i = 0; i < NA; ++i)
        {
            const int row = row0 + 32 * i;
            if (row >= rows)
                continue;
            const bool all = col + 12 <= p.N;
            uint32_t o[6];
#pragma unroll
            for (int j = 0; j < 3; ++j)
            {
                const f32x4 v = acc[i][j];
                if constexpr (OUT == OUT_GATED)
                    o[j] = bf_pair(seam_gate<false>(p.act, v[0], v[1]), seam_gate<false>(p.act, v[2], v[3]));
                else if constexpr (OUT == OUT_STORE)
                {
                    const bool sq = p.act == GEMM_ACT_RELU2;
                    o[2 * j] = bf_pair(sq ? seam_relu2(v[0]) : v[0], sq ? seam_relu2(v[1]) : v[1]);
                    o[2 * j + 1] = bf_pair(sq ? seam_relu2(v[2]) : v[2], sq ? seam_relu2(v[3]) : v[3]);
                }
                else if (col + 4 * j < p.N)
                    *reinterpret_cast<float4*>(c + ((int64_t) row * p.ldc + col + 4 * j) * 4) = make_float4(v[0], v[1], v[2], v[3]);
            }
            if constexpr (OUT == OUT_GATED)
            {
                uint32_t* to = reinterpret_cast<uint32_t*>(c + ((int64_t) row * p.ldc + (col >> 1)) * 2);
#pragma unroll
                for (int j = 0; j < 3; ++j)
                    if (all || col + 4 * j < p.N)
                        to[j] = o[j];
            }
            else if constexpr (OUT == OUT_STORE)
            {
                uint2* to = reinterpret_cast<uint2*>(c + ((int64_t) row * p.ldc + col) * 2);
#pragma unroll
                for (int j = 0; j < 3; ++j)
                    if (all || col + 4 * j < p.N)
                        to[j] = make_uint2(o[2 * j], o[2 * j + 1]);
            }
        }
    }
};
namespace tall
{
// (named like the other two, 32 WM MT rows x 32 WN NT columns)
template <int WT, int WM, int WN, int MT, int NT, int OUT>
__global__ __launch_bounds__(64 * WAVES) void gemm_glds_kernel(const GemmParams p)
{
    static_assert(WT == W_BF16 && 32 * WM * MT == TALL_BM && 32 * WN * NT == TALL_BN, "one shape");
    extern __shared__ __attribute__((aligned(16))) char wide_lds[];
    const GroupTile gt = group_tile<TALL_BM>(p, (p.N + TALL_BN - 1) / TALL_BN, blockIdx.x);
    if (gt.group < 0)
        return; // behind the last tile
    const int first = p.group_off[gt.group], rows = p.group_off[gt.group + 1] - first;
    const int tiles_m = (rows + TALL_BM - 1) / TALL_BM, tn = gt.tile / tiles_m, height = ((rows + tiles_m - 1) / tiles_m + 31) / 32 * 32;
    const int m0 = (gt.tile - tn * tiles_m) * height, n0 = tn * TALL_BN;
    if (m0 >= rows)
        return; // (many rows, rounded up to whole steps)
    const int blocks = (min(height, rows - m0) + 31) / 32; // of a wave
    TallTile t;
    t.lane = threadIdx.x & 63;
    t.wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    t.lds = (uint32_t) (uintptr_t) (lds_ptr*) wide_lds;
    t.nt = p.K / 64;
    t.a = reinterpret_cast<const char*>(p.a);
    t.w = reinterpret_cast<const char*>(p.w) + gt.group * p.batch_w;
    const int row8 = t.wid * 8 + (t.lane >> 3), piece = t.lane & 7;
#pragma unroll
    for (int i = 0; i < 5; ++i)
    {
        const int row = i * 64 + row8, m = m0 + row;
        int r = first + (m < rows ? m : rows - 1);
        if (p.a_rows)
            r = p.a_rows[r];
        t.ao[i] = (uint32_t) r * (uint32_t) (p.lda * 2) + ((piece ^ a_swz(row)) << 4);
    }
#pragma unroll
    for (int i = 0; i < 3; ++i)
    {
        const int row = i * 64 + row8, col = n0 + row, n = col < p.N ? col : p.N - 1;
        t.wo[i] = (uint32_t) n * (uint32_t) p.ldw + ((piece ^ tall_w_swz(row)) << 4);
    }
    char* c = reinterpret_cast<char*>(p.c) + first * p.ldc * (OUT == OUT_FP32 ? 4 : 2);
    const int row0 = m0 + 16 * (t.wid >> 2) + (t.lane & 15), col = n0 + 48 * (t.wid & 3) + 12 * (t.lane >> 4);
    auto go = [&](auto na) {
        constexpr int NA = decltype(na)::value;
        t.run<NA>();
        t.leave<OUT, NA>(p, c, row0, col, rows);
    };
    switch (blocks)
    {
    case 9: return go(std::integral_constant<int, 9>());
    case 8: return go(std::integral_constant<int, 8>());
    case 7: return go(std::integral_constant<int, 7>());
    case 6: return go(std::integral_constant<int, 6>());
    case 5: return go(std::integral_constant<int, 5>());
    case 4: return go(std::integral_constant<int, 4>());
    default: return go(std::integral_constant<int, 3>());
    }
}
} // namespace tall
template <int OUT>
int launch_tall_out(const GemmParams& p, hipStream_t stream)
{
    const auto kernel = tall::gemm_glds_kernel<W_BF16, 9, 6, 1, 1, OUT>;
    launch_util::ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), TALL_LDS);
    const int64_t tiles = (p.group_total / TALL_BM + std::min<int64_t>(p.batch, p.group_total)) * ((p.N + TALL_BN - 1) / TALL_BN);
    hipLaunchKernelGGL(kernel, dim3((unsigned) tiles), dim3(64 * WAVES), TALL_LDS, stream, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
    {
        set_error("gemm tall tiles: launch failed: %s", hipGetErrorString(e));
        return -1;
    }
    return 0;
}
// p: serves<W_BF16>(p); two K-tiles at least (the rule that picks them asks for eight)
inline bool tall_serves(const GemmParams& p)
{
    return p.K >= 128 && p.group_off && !p.resid && !p.bias && p.seam.n_sec == 0 && (p.act == GEMM_ACT_NONE || p.act == GEMM_ACT_RELU2 || p.act >= GEMM_ACT_GATE_SILU) && (p.out_dtype == DT_BFLOAT16 || p.act == GEMM_ACT_NONE);
}
// p: tall_serves(p)
inline int launch_tall(const GemmParams& p, hipStream_t stream)
{
    return p.act >= GEMM_ACT_GATE_SILU ? launch_tall_out<OUT_GATED>(p, stream) : p.out_dtype == DT_FLOAT ? launch_tall_out<OUT_FP32>(p, stream) : launch_tall_out<OUT_STORE>(p, stream);
}

inline bool aligned16(const void* p)
{
    return !(reinterpret_cast<uintptr_t>(p) & 15);
}

// what the kernel takes: everything that leaves does so in whole 16-byte pieces
template <int WT>
bool serves(const GemmParams& p)
{
    constexpr int ES = WT == W_INT8_SQ ? 1 : 2;
    if (p.wtype != WT || p.K <= 0 || (p.K * ES) % 128 || !aligned16(p.a) || !aligned16(p.w) || (p.lda * ES) % 16 || p.ldw % 16)
        return false;
    const GemmSection* last = WT == W_BF16 && p.seam.n_sec > 0 ? &p.seam.sec[p.seam.n_sec - 1] : nullptr;
    if (p.N % 8 && (!last || last->col0 > p.N - p.N % 8 || !last->f32 || p.bias)) // (columns that are no whole piece: one by one, in the last section)
        return false;
    // 32-bit offsets of the operands' rows (gathered rows: any of the a that the caller has; its extent is not known here)
    const int64_t rows = p.group_off ? p.group_total : p.M;
    if (rows * p.lda * ES >= (1ll << 31) || (int64_t) p.N * p.ldw >= (1ll << 31))
        return false;
    if constexpr (WT == W_BF16)
    {
        const int c_es = p.out_dtype == DT_FLOAT ? 4 : 2;
        if (p.batch > 1 && (p.batch_a % 16 || p.batch_w % 16 || p.batch_c % 16))
            return false;
        if (p.resid)
            return aligned16(p.resid) && p.ldr % 4 == 0 && (!p.gate || (aligned16(p.gate) && p.ldg % 8 == 0 && aligned16(p.gate_bias)));
        if ((p.out_dtype != DT_BFLOAT16 && p.out_dtype != DT_FLOAT) || !aligned16(p.bias) || (p.act != GEMM_ACT_NONE && p.act != GEMM_ACT_RELU2 && p.act < GEMM_ACT_GATE_SILU))
            return false;
        const bool gated = p.act >= GEMM_ACT_GATE_SILU;
        if ((p.seam.n_sec == 0 || p.seam.sec[0].col0 > 0)
            && (!aligned16(p.c) || p.ldc % (gated ? 8 : 16 / c_es) || (gated && p.out_dtype != DT_BFLOAT16)))
            return false;
        for (int s = 0; s < p.seam.n_sec; ++s)
        {
            const GemmSection& k = p.seam.sec[s];
            if (k.col0 % 8 || (k.act != GEMM_ACT_NONE && k.act != GEMM_ACT_RELU2))
                return false;
            if ((!k.f32 || k.act != GEMM_ACT_NONE) && (p.N % 8 || !aligned16(k.c) || k.ldc % (k.f32 ? 4 : 8)))
                return false;
        }
        return true;
    }
    else
    {
        const bool dual = WT == W_INT8_SQ && p.w2;
        if (p.out_dtype != DT_HALF && !dual)
            return false;
        if (p.ldc % 8 || reinterpret_cast<uintptr_t>(p.c) % (dual ? 8 : 16) || (p.residual && (dual || !aligned16(p.residual))) || (p.silu_gate && (WT != W_FP16 || p.residual || !aligned16(p.silu_gate))))
            return false;
        if constexpr (WT == W_INT8_SQ)
            return p.scale_col && p.scale_row && (!p.per_channel || aligned16(p.scale_col))
                && (!dual || (p.scale_col2 && p.swiglu_qscale && !p.per_token && aligned16(p.w2) && (!p.per_channel || aligned16(p.scale_col2))));
        return true;
    }
}

// at most this many tiles (grouped: full ones, and one begun in every group that has rows)
inline int64_t most_tiles(const GemmParams& p)
{
    const int of_tile = p.wtype == W_INT8_SQ && p.w2 ? BN / 2 : BN;
    const int64_t cols = (p.N + of_tile - 1) / of_tile;
    if (p.group_off)
        return (p.group_total / BM + std::min<int64_t>(p.batch, p.group_total)) * cols;
    return (int64_t) ((p.M + BM - 1) / BM) * cols * p.batch;
}

// What a plain or batched product costs on these tiles, in K-tiles of a lock-step 256 x 256 tile on a full chip (1.77 us each): the fewer CUs have one, the
// faster they run (their common power and L2; 1.2 us a K-tile with 128 of 256, 1.36 with 192, 1.5 with all), and the launch, its first requests and the results
// take the time of eight.  A tile of up to 128 rows costs two thirds.
inline double cost(const GemmParams& p, int es)
{
    const double tiles = (double) most_tiles(p), cus = launch_util::device_cus(), rounds = std::ceil(tiles / cus), fill = tiles / rounds / cus;
    return rounds * ((double) ((int64_t) p.K * es / 128) * (0.56 + 0.29 * fill) * (p.M <= BM / 2 ? 0.65 : 1.0) + 1.0) + 7.0;
}

template <int WT, int OUT, bool GROUPED = false>
int launch_out(const GemmParams& p, hipStream_t stream)
{
    const auto kernel = wide_kernel<WT, OUT, GROUPED>;
    launch_util::ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), LDS_BYTES);
    const int64_t tiles = most_tiles(p), cus = launch_util::device_cus(), rounds = (tiles + cus - 1) / cus;
    // even rounds: no workgroup has more than one tile more than another, and where some CUs have nothing to do the others run faster.  Grouped: a tile a
    // workgroup, as tiles of few rows and of many follow one another (in rounds the same within 2 %)
    const int64_t grid = GROUPED ? tiles : (tiles + rounds - 1) / rounds;
    hipLaunchKernelGGL(kernel, dim3((unsigned) grid), dim3(64 * WAVES), LDS_BYTES, stream, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
    {
        set_error("gemm_wide launch failed: %s", hipGetErrorString(e));
        return -1;
    }
    return 0;
}

// p: serves<WT>(p)
template <int WT>
int launch(const GemmParams& p, hipStream_t stream)
{
    if constexpr (WT == W_BF16)
    {
        const bool gated = p.act >= GEMM_ACT_GATE_SILU, fp32 = p.out_dtype == DT_FLOAT && p.seam.n_sec == 0 && p.act == GEMM_ACT_NONE;
        if (p.group_off)
            return gated ? launch_out<WT, OUT_GATED, true>(p, stream) : fp32 ? launch_out<WT, OUT_FP32, true>(p, stream) : launch_out<WT, OUT_STORE, true>(p, stream);
        if (p.resid)
            return p.gate ? launch_out<WT, OUT_RESID_GATE>(p, stream) : launch_out<WT, OUT_RESID>(p, stream);
        return gated ? launch_out<WT, OUT_GATED>(p, stream) : fp32 ? launch_out<WT, OUT_FP32>(p, stream) : launch_out<WT, OUT_STORE>(p, stream);
    }
    else if constexpr (WT == W_INT8_SQ)
        return p.w2 ? launch_out<WT, OUT_DUAL>(p, stream) : launch_out<WT, OUT_HALF>(p, stream);
    else
        return launch_out<WT, OUT_HALF>(p, stream);
}

template <int WT, int OUT, bool GROUPED, int WM, int WN, int MT, int NT, int S, bool PINNED>
int launch_row128_out(const GemmParams& p, hipStream_t stream)
{
    constexpr int BM = WM * MT * 32, BN = WN * NT * 32;
    constexpr size_t lds = (size_t) S * (BM + BN) * 128;
    static_assert(BM == 128 && lds <= LDS_BYTES, "LDS");
    const auto kernel = gemm_glds_kernel<WT, WM, WN, MT, NT, S, OUT, GROUPED, PINNED>;
    launch_util::ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), lds);
    const int64_t cols = (p.N + BN - 1) / BN;
    // grouped: at most this many row tiles, full ones, and one begun in every group that has rows
    const int64_t tiles = GROUPED ? (p.group_total / BM + std::min<int64_t>(p.batch, p.group_total)) * cols : (p.M + BM - 1) / BM * cols;
    hipLaunchKernelGGL(kernel, dim3((unsigned) tiles, GROUPED || WT != W_BF16 ? 1 : p.batch), dim3(64 * WM * WN), lds, stream, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
    {
        set_error("gemm tiles of 128 rows: launch failed: %s", hipGetErrorString(e));
        return -1;
    }
    return 0;
}
// p: serves<W_BF16>(p)
template <int WM, int WN, int MT, int NT, int S, bool PINNED>
int launch_row128(const GemmParams& p, hipStream_t stream)
{
    const bool gated = p.act >= GEMM_ACT_GATE_SILU, fp32 = p.out_dtype == DT_FLOAT && p.seam.n_sec == 0 && p.act == GEMM_ACT_NONE;
    if (p.group_off)
        return gated ? launch_row128_out<W_BF16, OUT_GATED, true, WM, WN, MT, NT, S, PINNED>(p, stream)
            : fp32   ? launch_row128_out<W_BF16, OUT_FP32, true, WM, WN, MT, NT, S, PINNED>(p, stream)
                     : launch_row128_out<W_BF16, OUT_STORE, true, WM, WN, MT, NT, S, PINNED>(p, stream);
    if (p.resid)
        return p.gate ? launch_row128_out<W_BF16, OUT_RESID_GATE, false, WM, WN, MT, NT, S, PINNED>(p, stream) : launch_row128_out<W_BF16, OUT_RESID, false, WM, WN, MT, NT, S, PINNED>(p, stream);
    return gated ? launch_row128_out<W_BF16, OUT_GATED, false, WM, WN, MT, NT, S, PINNED>(p, stream)
        : fp32   ? launch_row128_out<W_BF16, OUT_FP32, false, WM, WN, MT, NT, S, PINNED>(p, stream)
                 : launch_row128_out<W_BF16, OUT_STORE, false, WM, WN, MT, NT, S, PINNED>(p, stream);
}

} // namespace wide
} // namespace
} // namespace kernels
} // namespace tllm
