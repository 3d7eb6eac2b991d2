// Attention of the stack engine over the paged cache: the MFMA tile kernel for bfloat16 (prefill portions and decoded tokens
// alike), and the dispatch between it and the general kernel of stack_ops.hip (any shape, both element types).
//
// attn_tile_kernel: one workgroup per (16 rows of one entry, head); its NW waves split the key blocks (32 keys each) round-robin -
// key-split waves, so a decoded token with a long context still has NW waves in flight - and merge their partial (max, sum, O)
// through LDS.  Everything is computed TRANSPOSED so that no operand ever changes layout between the two products:
//   S^T = K Q^T      A = K rows straight from the page (key-major, 16 bytes of dim per lane), B = Q^T fragments kept in registers;
//                    the result has one query row per lane column, 4 keys per lane and tile;
//   O^T += V^T P^T   B = P^T, which is exactly what the lane already holds (its 8 scores of the block, as bfloat16);
//                    A = V^T rows, which is why the cache stores values channel-major inside a page ([vdim][page]).
// Both maps of a differential head run side by side and share the V^T fragments.  fp32: scores, soft cap, softmax state, O.
#include "dev_utils.h"
#include "launch_util.h"
#include "stack_attn_order.h"
#include "stack_kernels.h"
#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace tllm
{
namespace kernels
{
int launch_stack_attention_general(const StackAttnParams& p, hipStream_t stream); // stack_ops.hip

using namespace dev;

namespace
{
constexpr int kSplitRows = 64, kMaxSplits = 16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4))); // staging registers: arrays of HIP's uint4 end up in scratch memory

__device__ __forceinline__ bf16x8 as_bf16x8(const uint4& u)
{
    bf16x8 r;
    __builtin_memcpy(&r, &u, 16);
    return r;
}

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

// max / sum over the four lanes that hold the same query row (lane ^ 16, lane ^ 32)
__device__ __forceinline__ float rows_max(float v)
{
    v = fmaxf(v, __shfl_xor(v, 16, 64));
    return fmaxf(v, __shfl_xor(v, 32, 64));
}
__device__ __forceinline__ float rows_sum(float v)
{
    v += __shfl_xor(v, 16, 64);
    return v + __shfl_xor(v, 32, 64);
}

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{lo, hi}, bf16x2_t));
}

// What a head does to its raw scores, in the base-2 domain (an exponential is one v_exp_f32, a logarithm one v_log_f32):
//   score2 = cap(q.k * scale) * temp * log2 e - slope2 * (i - j) - r1 * log2(1 + r2 * (i - j))
// and how scores become weights: softmax (running maximum and sum), or a sigmoid per key (no state across keys).
struct HeadMods
{
    float scale2, cap2, cap_arg, temp, slope2, r1, r2, wb2;
    int pen, sigm; // pen: any of temp / slope / r1 is set
    int keep;      // the first `keep` keys of the sequence stay visible behind a window
};

// Which query, key and value head a launch's head index h stands for.  Ordinarily h is the query head and reads the key / value head
// of its group.  cross_values: p.heads = query heads x kv_heads, and h = query head * kv_heads + value head - every query head's
// weights applied to every value head's rows (the terms a mixing of weights across heads is made of).
struct HeadMap
{
    int qh, kh, vh, q_heads;
};
__device__ __forceinline__ HeadMap head_map(const StackAttnParams& p, int h)
{
    HeadMap m;
    m.q_heads = p.cross_values ? p.heads / p.kv_heads : p.heads;
    m.qh = p.cross_values ? h / p.kv_heads : h;
    m.kh = m.qh / (m.q_heads / p.kv_heads);
    m.vh = p.cross_values ? h % p.kv_heads : m.kh;
    return m;
}

__device__ __forceinline__ HeadMods head_mods(const StackAttnParams& p, int h)
{
    constexpr float LOG2E = 1.4426950408889634f;
    h = p.cross_values ? h / p.kv_heads : h; // per-head numbers belong to query heads
    HeadMods m;
    m.temp = p.temp ? p.temp[h] : 1.f;
    m.scale2 = p.scale * LOG2E * (p.softcap > 0.f ? 1.f : m.temp);
    m.cap2 = p.softcap > 0.f ? p.softcap * LOG2E * m.temp : 0.f;
    m.cap_arg = p.softcap > 0.f ? p.scale / p.softcap * 2.f * LOG2E : 0.f;
    m.slope2 = p.slope ? p.slope[h] * LOG2E : 0.f;
    m.r1 = p.log_r1 ? p.log_r1[h] : 0.f;
    m.r2 = p.log_r1 ? p.log_r2[h] : 0.f;
    m.pen = (p.slope || p.log_r1) ? 1 : 0;
    m.sigm = p.weights == WEIGHTS_SIGMOID;
    m.wb2 = m.sigm && p.wbias ? p.wbias[h] * LOG2E : 0.f;
    m.keep = p.mask == MASK_WINDOW ? p.mask_keep : 0;
    return m;
}

// the first key position a row at `pos` sees
__device__ __forceinline__ int first_visible(const StackAttnParams& p, int pos)
{
    if (p.mask == MASK_WINDOW)
        return pos - p.mask_size + 1 > 0 ? pos - p.mask_size + 1 : 0;
    if (p.mask == MASK_CHUNK)
        return pos / p.mask_size * p.mask_size;
    return 0;
}

// The 32-key blocks a tile walks: from the block that holds its first row's first visible key up to the block of its last row;
// with kept first keys, the blocks that hold them and lie before that range come first.  Step v of n visits block walk_block(w, v).
struct BlockWalk
{
    int nkeep, lo, n;
};
__device__ __forceinline__ BlockWalk block_walk(const StackAttnParams& p, int first_row_pos, int nblk)
{
    BlockWalk w;
    w.lo = first_visible(p, first_row_pos) / 32;
    const int kept = (p.mask == MASK_WINDOW && p.mask_keep > 0) ? (p.mask_keep + 31) / 32 : 0;
    w.nkeep = kept < w.lo ? kept : w.lo;
    w.n = w.nkeep + (nblk - w.lo);
    return w;
}
__device__ __forceinline__ int walk_block(const BlockWalk& w, int v)
{
    return v < w.nkeep ? v : v - w.nkeep + w.lo;
}

// Scores of one 32-key block of one map -> its P^T fragment, with the online-softmax state of the lane's query row brought up to
// date.  `masked` is wave-uniform: only blocks that reach past the first row's position, or start before the last row's first
// visible key, compare keys with positions.  Each option is one branch around its eight scores: with the options tested score by score the
// loop held two scalar branches per score and option, and the code of options that a model does not have was fetched all the same (attn_tile_kernel of
// two maps of 64 x 128 14.9 KB, 10.2 this way with the split form on its own; prompts of latent keys 320 x 256, 1021 rows 58.4 -> 49.5 us, 2048 rows
// 110.9 -> 94.7, three of 1021 rows in the wide form 189.9 -> 163.4).
template <int VT>
__device__ __forceinline__ uint4 softmax_block(f32x4 (&s)[2], float& m_run, float& l_run, f32x4 (&acc)[VT], const HeadMods& hm, bool masked,
    int key_lane0, int qpos, int klo)
{
#define EACH_SCORE _Pragma("unroll") for (int t = 0; t < 2; ++t) _Pragma("unroll") for (int i = 0; i < 4; ++i)
    if (hm.cap2 > 0.f)
    {
        // cap * tanh(x / cap) with tanh(y) = (e^{2y} - 1) / (e^{2y} + 1); cap_arg = scale / cap * 2 log2 e
        EACH_SCORE
        {
            const float t2 = __builtin_amdgcn_exp2f(fminf(fmaxf(s[t][i] * hm.cap_arg, -43.f), 43.f));
            s[t][i] = hm.cap2 * (t2 - 1.f) * __builtin_amdgcn_rcpf(t2 + 1.f);
        }
    }
    else
        EACH_SCORE s[t][i] *= hm.scale2;
    if (hm.pen)
    {
        EACH_SCORE s[t][i] -= hm.slope2 * (float) (qpos - (key_lane0 + t * 16 + i));
        if (hm.r1 != 0.f)
            EACH_SCORE s[t][i] -= hm.r1 * __builtin_amdgcn_logf(fmaxf(1.f + hm.r2 * (float) (qpos - (key_lane0 + t * 16 + i)), 1e-30f));
    }
    if (masked)
        EACH_SCORE
        {
            const int kidx = key_lane0 + t * 16 + i;
            if (kidx > qpos || (kidx < klo && kidx >= hm.keep))
                s[t][i] = -INFINITY;
        }
    float bm = -INFINITY;
    EACH_SCORE bm = fmaxf(bm, s[t][i]);
#undef EACH_SCORE
    if (hm.sigm)
    {
        // every key's weight stands alone: 1 / (1 + 2^-(score2 + offset2)); a hidden key's is 2^-inf = 0
        float pv[8];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                pv[t * 4 + i] = s[t][i] == -INFINITY ? 0.f : __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-(s[t][i] + hm.wb2)));
        return make_uint4(pack_bf16(pv[0], pv[1]), pack_bf16(pv[2], pv[3]), pack_bf16(pv[4], pv[5]), pack_bf16(pv[6], pv[7]));
    }
    bm = rows_max(bm);
    const float mn = fmaxf(m_run, bm);
    const bool none = mn == -INFINITY; // this row sees no key of this block (nor of any before)
    const float corr = none ? 1.f : __builtin_amdgcn_exp2f(m_run - mn);
    float rs = 0.f, pv[8];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
        {
            pv[t * 4 + i] = none ? 0.f : __builtin_amdgcn_exp2f(s[t][i] - mn);
            rs += pv[t * 4 + i];
        }
    l_run = l_run * corr + rs; // (the lane's own keys: the four lanes of a row share its maximum, their sums meet behind the last block)
    m_run = mn;
    // the accumulators are rescaled only when some row's maximum moved (wave-uniform test): behind the first blocks of a long
    // context it rarely does, and the accumulators sit in the matrix pipe's registers, a round trip per element away
    if (__builtin_amdgcn_ballot_w64(corr != 1.f) != 0)
    {
#pragma unroll
        for (int ct = 0; ct < VT; ++ct)
            acc[ct] *= corr;
    }
    return make_uint4(pack_bf16(pv[0], pv[1]), pack_bf16(pv[2], pv[3]), pack_bf16(pv[4], pv[5]), pack_bf16(pv[6], pv[7]));
}

// How a finished row leaves: the softmax denominator also takes the head's sink (a logit without key or value), given the row's
// running maximum M (base 2) and sum L relative to it -> the factor on the accumulator; sigmoid weights are not normalised.
__device__ __forceinline__ float finish_factor(const StackAttnParams& p, int h, float M, float L)
{
    if (p.weights == WEIGHTS_SIGMOID)
        return 1.f;
    if (!p.sink)
        return 1.f / L;
    const float sk = p.sink[p.cross_values ? h / p.kv_heads : h] * 1.4426950408889634f, mf = fmaxf(M, sk);
    const float wk = __builtin_amdgcn_exp2f(M - mf);
    return wk / (L * wk + __builtin_amdgcn_exp2f(sk - mf));
}

__device__ __forceinline__ float out_gate_of(const StackAttnParams& p, int64_t t, int h)
{
    if (!p.out_gate)
        return 1.f;
    const float z = bf2f(reinterpret_cast<const uint16_t*>(p.out_gate)[t * p.ld_gate + h]);
    return 1.f / (1.f + __expf(-z));
}

template <int MAPS, int DK, int VT, int NW, bool SPLIT>
__global__ __launch_bounds__(NW * 64, 3 * MAPS * DK + (1 + MAPS) * VT <= 42 ? 2 : 1) void attn_tile_kernel(const StackAttnParams p, int below_count, int ks, int head_rows)
{
    // VP: 16 floats behind a row's channels put the 16 rows x 4 pieces that a wave stores at once on all banks alike.  (Rows of V floats, a
    // float per store, met on one bank 16 at a time: one decoded token took 10.7 us with two maps of 64 x 128 at 154 keys, 13.7 us with
    // latent keys of 320 x 256 under a window of 512; 8.1 and 11.5 us this way.)  SPLIT is the instance of ks > 1: a launch of few cycles is bound by
    // fetching its code, and each form carried the other's end.  Two waves per SIMD where the operands leave room: Q and two key tiles of every map (3 MAPS
    // DK), a value tile and the accumulators ((1 + MAPS) VT) take 4 registers each, and some 55 are needed beside them, so up to 42 x 4 fit 256 (one map of 192 x
    // 192: 222; two of 128 x 128, 48 x 4, want 254 and more).  That keeps the accumulators out of the accumulation registers, from which every block's
    // rescaling moved them back and forth (two maps of 64 x 128 8.3 -> 7.4 us, five requests of 300 keys 12.4 -> 11.5, one map of 128 x 128 in one round 5.9 -> 5.4; 192 x 128 in two splits 7.6 as before).
    constexpr int D = DK * 32, V = VT * 16, VP = V + 16;
    extern __shared__ float lds[];
    float* o_part = lds;                          // [NW][MAPS][16][VP]
    float* ml_part = lds + NW * MAPS * 16 * VP;    // [NW][MAPS][16][2]
    // Not SPLIT: blockIdx.x is the entry's 16-row tile.  SPLIT (ks > 1; decoding steps: every entry one tile): blockIdx.x is the key split -
    // workgroup `split` of an (entry, head) takes the key blocks split * NW + w, + ks * NW, ... and leaves an unnormalised partial
    // (max, sum, O per map and row) in split_ws; attn_split_merge_kernel finishes the rows.
    // head_rows (a step of single decoded tokens whose heads share key/value heads and have no numbers inside the score): the tile's 16
    // rows are up to 16 HEADS of one key/value head's group, at the entry's one token; blockIdx.z counts such sets of heads (head_rows of
    // them per key/value head) - the keys are walked once per set
    const int e = blockIdx.y, group = p.heads / p.kv_heads;
    const int hbase = head_rows ? blockIdx.z / head_rows * group + blockIdx.z % head_rows * 16 : 0, h = head_rows ? hbase : blockIdx.z;
    const int hend = head_rows ? min(hbase + 16, ((int) blockIdx.z / head_rows + 1) * group) : p.heads; // behind the set's last head
    const int r0 = (SPLIT || head_rows) ? 0 : blockIdx.x * 16;
    const int split = SPLIT ? blockIdx.x : 0;
    const int count = p.ent_count[e];
    if (r0 >= count || count >= below_count) // entries of below_count rows and more are the prefill form's
        return;
    const int first = p.ent_first[e], pos0 = p.ent_pos0[e];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int col = lane & 15, g4 = lane >> 4;
    const HeadMap hd = head_map(p, h);
    const int g = hd.kh, gv = hd.vh;
    const int page = p.page;
    const int32_t* table = p.block_table + (int64_t) e * p.max_blocks;
    const HeadMods hm = head_mods(p, h);
    const uint16_t* kp = reinterpret_cast<const uint16_t*>(p.k_pool);
    const uint16_t* vp = reinterpret_cast<const uint16_t*>(p.v_pool);

    const int qrow = head_rows ? 0 : (r0 + col < count ? r0 + col : count - 1);
    const int qhead = head_rows ? (hbase + col < hend ? hbase + col : hend - 1) : hd.qh;
    const int qpos = pos0 + qrow;
    const int klo = first_visible(p, qpos);
    bf16x8 qf[MAPS][DK];
#pragma unroll
    for (int m = 0; m < MAPS; ++m)
#pragma unroll
        for (int ks = 0; ks < DK; ++ks)
            qf[m][ks] = as_bf16x8(*reinterpret_cast<const uint4*>(
                reinterpret_cast<const uint16_t*>(p.q) + (((int64_t) (first + qrow) * hd.q_heads + qhead) * MAPS + m) * D + ks * 32 + 8 * g4));
    const int last_row = head_rows ? 0 : (r0 + 15 < count ? r0 + 15 : count - 1);
    const int nblk = (pos0 + last_row) / 32 + 1;
    // the tile's key blocks: from the one that holds the first row's first visible key; klo_last: the last row's (the largest)
    const int blk_lo = first_visible(p, pos0 + r0) / 32, klo_last = first_visible(p, pos0 + last_row);

    float m_run[MAPS], l_run[MAPS];
    f32x4 acc[MAPS][VT];
#pragma unroll
    for (int m = 0; m < MAPS; ++m)
    {
        m_run[m] = -INFINITY;
        l_run[m] = 0.f;
#pragma unroll
        for (int ct = 0; ct < VT; ++ct)
            acc[m][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // Software pipeline: the K fragments of a block are requested one iteration ahead, its V^T fragments at the top of its own
    // iteration, so that the score / softmax arithmetic of a block (the long part: it is all VALU) runs with both in flight.
    uint4 kf[MAPS][2][DK];
    auto request_k = [&](int kb, int blk) {
        const int off = (kb * 32) % page;
#pragma unroll
        for (int m = 0; m < MAPS; ++m)
#pragma unroll
            for (int t = 0; t < 2; ++t)
            {
                const uint16_t* krow = kp + (((int64_t) blk * (p.kv_heads * MAPS) + g * MAPS + m) * page + off + t * 16 + col) * D + 8 * g4;
#pragma unroll
                for (int ks = 0; ks < DK; ++ks)
                    kf[m][t][ks] = *reinterpret_cast<const uint4*>(krow + ks * 32);
            }
    };
    const BlockWalk bw = block_walk(p, pos0 + r0, nblk);
    const int vb0 = split * NW + w, kstep = SPLIT ? ks * NW : NW;
    int kb_next = vb0 < bw.n ? walk_block(bw, vb0) : 0;
    int blk = vb0 < bw.n ? table[kb_next * 32 / page] : 0;
    if (vb0 < bw.n)
        request_k(kb_next, blk);
    for (int vb = vb0; vb < bw.n; vb += kstep)
    {
        const int kb = kb_next;
        const int key0 = kb * 32, off = key0 % page;
        uint2 vlo[VT], vhi[VT];
        {
            const uint16_t* vrow = vp + (((int64_t) blk * p.kv_heads + gv) * V + col) * page + off + 4 * g4;
#pragma unroll
            for (int ct = 0; ct < VT; ++ct)
            {
                vlo[ct] = *reinterpret_cast<const uint2*>(vrow + (int64_t) ct * 16 * page);
                vhi[ct] = *reinterpret_cast<const uint2*>(vrow + (int64_t) ct * 16 * page + 16);
            }
        }
        f32x4 s[MAPS][2];
#pragma unroll
        for (int m = 0; m < MAPS; ++m)
#pragma unroll
            for (int t = 0; t < 2; ++t)
            {
                s[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < DK; ++ks)
                    s[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(kf[m][t][ks]), qf[m][ks], s[m][t], 0, 0, 0);
            }
        if (vb + kstep < bw.n)
        {
            kb_next = walk_block(bw, vb + kstep);
            blk = table[kb_next * 32 / page];
            request_k(kb_next, blk);
        }
        uint4 pf[MAPS]; // P^T fragment of the block, 8 bfloat16 per map
        const bool masked = key0 + 31 > pos0 + r0 || key0 < klo_last; // wave-uniform
#pragma unroll
        for (int m = 0; m < MAPS; ++m)
            pf[m] = softmax_block<VT>(s[m], m_run[m], l_run[m], acc[m], hm, masked, key0 + 4 * g4, qpos, klo);
        // O^T += V^T P^T: slot j of the lane's k group is key 4 g4 + j (j < 4) or 16 + 4 g4 + (j - 4) of the block, in both operands
#pragma unroll
        for (int ct = 0; ct < VT; ++ct)
        {
            const bf16x8 vf = as_bf16x8(make_uint4(vlo[ct].x, vlo[ct].y, vhi[ct].x, vhi[ct].y));
#pragma unroll
            for (int m = 0; m < MAPS; ++m)
                acc[m][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, as_bf16x8(pf[m]), acc[m][ct], 0, 0, 0);
        }
    }

    // ---- merge of the waves' partials
#pragma unroll
    for (int m = 0; m < MAPS; ++m)
    {
        l_run[m] = rows_sum(l_run[m]);
        if (g4 == 0)
        {
            ml_part[((w * MAPS + m) * 16 + col) * 2] = m_run[m];
            ml_part[((w * MAPS + m) * 16 + col) * 2 + 1] = l_run[m];
        }
#pragma unroll
        for (int ct = 0; ct < VT; ++ct)
            *reinterpret_cast<f32x4*>(&o_part[((w * MAPS + m) * 16 + col) * VP + ct * 16 + 4 * g4]) = acc[m][ct];
    }
    __syncthreads();
    // 16 threads per row at NW = 4 (NW * 4 in general), each a strided set of channels
    constexpr int TPR = NW * 4;
    const int row = threadIdx.x / TPR, sub = threadIdx.x % TPR;
    // where tile row `row` leaves: (packed row, head)
    const int64_t out_t = first + (head_rows ? 0 : r0 + row);
    const int out_h = head_rows ? hbase + row : h;
    const bool out_ok = head_rows ? hbase + row < hend : r0 + row < count;
    float wgt[MAPS][NW];
#pragma unroll
    for (int m = 0; m < MAPS; ++m)
    {
        float M = -INFINITY;
#pragma unroll
        for (int ww = 0; ww < NW; ++ww)
            M = fmaxf(M, ml_part[((ww * MAPS + m) * 16 + row) * 2]);
        float L = 0.f;
#pragma unroll
        for (int ww = 0; ww < NW; ++ww)
        {
            const float mw = ml_part[((ww * MAPS + m) * 16 + row) * 2];
            wgt[m][ww] = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - M); // the running maxima are base-2 exponents
            if (hm.sigm)
                wgt[m][ww] = 1.f; // sigmoid weights: the waves' sums simply add
            L += wgt[m][ww] * ml_part[((ww * MAPS + m) * 16 + row) * 2 + 1];
        }
        if constexpr (SPLIT)
        {
            // partial of this split: weights stay relative to the split's own maximum, nothing is divided yet
            if (sub == 0 && out_ok)
            {
                float* ws = p.split_ws + (((out_t * p.heads + out_h) * ks + split) * MAPS + m) * (V + 2);
                ws[V] = M;
                ws[V + 1] = L;
            }
        }
        else
        {
            const float fin = finish_factor(p, out_h < p.heads ? out_h : p.heads - 1, M, L);
#pragma unroll
            for (int ww = 0; ww < NW; ++ww)
                wgt[m][ww] *= fin;
        }
    }
    constexpr int CPT = (V + TPR - 1) / TPR;
    if constexpr (SPLIT)
    {
        if (out_ok)
        {
#pragma unroll
            for (int m = 0; m < MAPS; ++m)
            {
                float* ws = p.split_ws + (((out_t * p.heads + out_h) * ks + split) * MAPS + m) * (V + 2);
#pragma unroll
                for (int c = 0; c < CPT; ++c)
                {
                    const int ch = sub + c * TPR;
                    if (ch < V)
                    {
                        float a = 0.f;
#pragma unroll
                        for (int ww = 0; ww < NW; ++ww)
                            a += wgt[m][ww] * o_part[((ww * MAPS + m) * 16 + row) * VP + ch];
                        ws[ch] = a;
                    }
                }
            }
        }
        return;
    }
    float o[CPT], ss = 0.f;
#pragma unroll
    for (int c = 0; c < CPT; ++c)
    {
        const int ch = sub + c * TPR;
        o[c] = 0.f;
        if (ch < V)
        {
            float a[MAPS];
#pragma unroll
            for (int m = 0; m < MAPS; ++m)
            {
                a[m] = 0.f;
#pragma unroll
                for (int ww = 0; ww < NW; ++ww)
                    a[m] += wgt[m][ww] * o_part[((ww * MAPS + m) * 16 + row) * VP + ch];
            }
            o[c] = MAPS == 2 ? a[0] - p.lambda * a[MAPS - 1] : a[0];
            ss += o[c] * o[c];
        }
    }
    float mul = 1.f;
    if (p.head_norm)
    {
#pragma unroll
        for (int d = 1; d < TPR; d <<= 1)
            ss += __shfl_xor(ss, d, 64);
        mul = p.out_scale / sqrtf(ss / (float) V + p.eps);
    }
    if (out_ok)
    {
        mul *= out_gate_of(p, out_t, out_h);
        uint16_t* out = reinterpret_cast<uint16_t*>(p.out) + (out_t * p.heads + out_h) * V;
#pragma unroll
        for (int c = 0; c < CPT; ++c)
            if (sub + c * TPR < V)
                out[sub + c * TPR] = f2bf(o[c] * mul);
    }
}

// attn_prefill_kernel: the form for entries that bring many rows.  One workgroup per (64 rows of an entry, head), wave w owns rows
// 16 w .. 16 w + 15; all four waves walk the same 32-key blocks, which the workgroup stages once through LDS (K rows padded to an odd
// number of 16-byte pieces, V^T rows to 80 bytes: the fragment reads spread over the banks) - the next block's global loads are in
// flight while this block is computed.  Same transposed products and operand slots as attn_tile_kernel; no merge: a wave finishes
// its own rows (lambda combination, head norm, bfloat16 store).  Tiles are handed out heaviest first (the last rows see most keys).
// Two waves per SIMD where the registers allow it: with the whole file to one wave the compiler keeps the accumulators in the
// accumulation registers and moves all of them back and forth around every block's softmax.
template <int MAPS, int DK, int VT>
__global__ __launch_bounds__(256, DK >= 10 ? 1 : 2) void attn_prefill_kernel(const StackAttnParams p, int min_count)
{
    constexpr int D = DK * 32, V = VT * 16;
    constexpr int KP = D * 2 + 16, VP = 80;                 // LDS row pitches in bytes
    constexpr int K16 = MAPS * 32 * (D / 8), V16 = V * 4;   // 16-byte pieces per block
    constexpr int KPT = (K16 + 255) / 256, VPT = (V16 + 255) / 256;
    __shared__ __attribute__((aligned(16))) char k_s[MAPS * 32 * KP];
    __shared__ __attribute__((aligned(16))) char v_s[V * VP];
    const int e = blockIdx.y, h = blockIdx.z;
    const int count = p.ent_count[e];
    if (count < min_count)
        return;
    const int tile = (count + 63) / 64 - 1 - (int) blockIdx.x;
    if (tile < 0)
        return;
    const int first = p.ent_first[e], pos0 = p.ent_pos0[e];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int col = lane & 15, g4 = lane >> 4;
    const HeadMap hd = head_map(p, h);
    const int g = hd.kh, gv = hd.vh;
    const int page = p.page;
    const int32_t* table = p.block_table + (int64_t) e * p.max_blocks;
    const HeadMods hm = head_mods(p, h);
    const uint16_t* kp = reinterpret_cast<const uint16_t*>(p.k_pool);
    const uint16_t* vp = reinterpret_cast<const uint16_t*>(p.v_pool);

    const int r0 = tile * 64 + w * 16;
    const bool wave_rows = r0 < count; // wave-uniform
    const int qrow = r0 + col < count ? r0 + col : count - 1;
    const int qpos = pos0 + qrow;
    const int klo = first_visible(p, qpos);
    bf16x8 qf[MAPS][DK];
#pragma unroll
    for (int m = 0; m < MAPS; ++m)
#pragma unroll
        for (int ks = 0; ks < DK; ++ks)
            qf[m][ks] = as_bf16x8(*reinterpret_cast<const uint4*>(
                reinterpret_cast<const uint16_t*>(p.q) + (((int64_t) (first + qrow) * hd.q_heads + hd.qh) * MAPS + m) * D + ks * 32 + 8 * g4));
    const int wg_last = tile * 64 + 63 < count ? tile * 64 + 63 : count - 1;
    const int nblk = (pos0 + wg_last) / 32 + 1;
    const int my_last = r0 + 15 < count ? r0 + 15 : count - 1;
    const int my_blk = wave_rows ? (pos0 + my_last) / 32 : -1; // the wave's last block that holds a visible key
    // ... and its first, and the workgroup's first (a window or a chunk hides everything before it)
    const int my_lo = wave_rows ? first_visible(p, pos0 + r0) / 32 : 0, klo_last = wave_rows ? first_visible(p, pos0 + my_last) : 0;
    const int wg_lo = first_visible(p, pos0 + tile * 64) / 32;

    float m_run[MAPS], l_run[MAPS];
    f32x4 acc[MAPS][VT];
#pragma unroll
    for (int m = 0; m < MAPS; ++m)
    {
        m_run[m] = -INFINITY;
        l_run[m] = 0.f;
#pragma unroll
        for (int ct = 0; ct < VT; ++ct)
            acc[m][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    u32x4 kr[KPT], vr[VPT];
    // the page id of a block is fetched one block before its rows are requested: one memory latency per block, not two in a row
    const BlockWalk bw = block_walk(p, pos0 + tile * 64, nblk);
    // blocks below this index hold kept first keys, which every row sees whatever its own window (a wave whose rows start further
    // down than the workgroup's first takes part in them too)
    const int keep_blk = (p.mask == MASK_WINDOW && p.mask_keep > 0) ? (p.mask_keep + 31) / 32 : 0;
    int blk_next = table[walk_block(bw, 0) * 32 / page];
    auto request = [&](int vb) {
        const int key0 = walk_block(bw, vb) * 32;
        const int blk = blk_next, off = key0 % page;
        blk_next = table[vb + 1 < bw.n ? walk_block(bw, vb + 1) * 32 / page : key0 / page];
#pragma unroll
        for (int i = 0; i < KPT; ++i)
        {
            const int idx = tid + i * 256;
            if (K16 % 256 == 0 || idx < K16)
            {
                const int row = idx / (D / 8), piece = idx % (D / 8); // row = map * 32 + key
                kr[i] = *reinterpret_cast<const u32x4*>(
                    kp + (((int64_t) blk * (p.kv_heads * MAPS) + g * MAPS + row / 32) * page + off + row % 32) * D + piece * 8);
            }
        }
#pragma unroll
        for (int i = 0; i < VPT; ++i)
        {
            const int idx = tid + i * 256;
            if (V16 % 256 == 0 || idx < V16)
                vr[i] = *reinterpret_cast<const u32x4*>(vp + (((int64_t) blk * p.kv_heads + gv) * V + idx / 4) * page + off + (idx % 4) * 8);
        }
    };
    request(0);
    for (int vb = 0; vb < bw.n; ++vb)
    {
        const int kb = walk_block(bw, vb);
#pragma unroll
        for (int i = 0; i < KPT; ++i)
        {
            const int idx = tid + i * 256;
            if (K16 % 256 == 0 || idx < K16)
                *reinterpret_cast<u32x4*>(k_s + (idx / (D / 8)) * KP + (idx % (D / 8)) * 16) = kr[i];
        }
#pragma unroll
        for (int i = 0; i < VPT; ++i)
        {
            const int idx = tid + i * 256;
            if (V16 % 256 == 0 || idx < V16)
                *reinterpret_cast<u32x4*>(v_s + (idx / 4) * VP + (idx % 4) * 16) = vr[i];
        }
        __syncthreads();
        if (vb + 1 < bw.n)
            request(vb + 1);
        if (kb <= my_blk && (kb >= my_lo || kb < keep_blk))
        {
            const int key0 = kb * 32;
            uint4 pf[MAPS];
            const bool masked = key0 + 31 > pos0 + r0 || key0 < klo_last; // wave-uniform
#pragma unroll
            for (int m = 0; m < MAPS; ++m)
            {
                f32x4 s[2];
#pragma unroll
                for (int t = 0; t < 2; ++t)
                {
                    s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int ks = 0; ks < DK; ++ks)
                        s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            as_bf16x8(*reinterpret_cast<const uint4*>(k_s + (m * 32 + t * 16 + col) * KP + (ks * 32 + 8 * g4) * 2)), qf[m][ks], s[t],
                            0, 0, 0);
                }
                pf[m] = softmax_block<VT>(s, m_run[m], l_run[m], acc[m], hm, masked, key0 + 4 * g4, qpos, klo);
            }
#pragma unroll
            for (int ct = 0; ct < VT; ++ct)
            {
                const char* vrow = v_s + (ct * 16 + col) * VP + 8 * g4;
                const uint2 lo = *reinterpret_cast<const uint2*>(vrow);
                const uint2 hi = *reinterpret_cast<const uint2*>(vrow + 32);
                const bf16x8 vf = as_bf16x8(make_uint4(lo.x, lo.y, hi.x, hi.y));
#pragma unroll
                for (int m = 0; m < MAPS; ++m)
                    acc[m][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, as_bf16x8(pf[m]), acc[m][ct], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    if (!wave_rows)
        return;
    // lane (col, g4) holds, for row col, channels ct * 16 + 4 g4 + i
    float inv[MAPS];
#pragma unroll
    for (int m = 0; m < MAPS; ++m)
        inv[m] = finish_factor(p, h, m_run[m], rows_sum(l_run[m]));
    float ss = 0.f;
#pragma unroll
    for (int ct = 0; ct < VT; ++ct)
#pragma unroll
        for (int i = 0; i < 4; ++i)
        {
            float o = acc[0][ct][i] * inv[0];
            if (MAPS == 2)
                o -= p.lambda * (acc[MAPS - 1][ct][i] * inv[MAPS - 1]);
            acc[0][ct][i] = o;
            ss += o * o;
        }
    float mul = 1.f;
    if (p.head_norm)
    {
        ss += __shfl_xor(ss, 16, 64);
        ss += __shfl_xor(ss, 32, 64);
        mul = p.out_scale / sqrtf(ss / (float) V + p.eps);
    }
    if (r0 + col < count)
    {
        mul *= out_gate_of(p, first + r0 + col, h);
        uint16_t* out = reinterpret_cast<uint16_t*>(p.out) + ((int64_t) (first + r0 + col) * p.heads + h) * V + 4 * g4;
#pragma unroll
        for (int ct = 0; ct < VT; ++ct)
            *reinterpret_cast<uint2*>(out + ct * 16) = make_uint2((uint32_t) f2bf(acc[0][ct][0] * mul) | ((uint32_t) f2bf(acc[0][ct][1] * mul) << 16),
                (uint32_t) f2bf(acc[0][ct][2] * mul) | ((uint32_t) f2bf(acc[0][ct][3] * mul) << 16));
    }
}

// the largest of a value over the lanes 16, 32 and 48 further on, without the LDS crossbar: a half's and a row's values change places
// (v_permlane32_swap, v_permlane16_swap: the two results together hold both partners' values)
__device__ __forceinline__ float rows_max_swap(float v)
{
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    const auto h = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const uint32_t x = __builtin_bit_cast(uint32_t, fmaxf(__builtin_bit_cast(float, (uint32_t) h[0]), __builtin_bit_cast(float, (uint32_t) h[1])));
    const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    return fmaxf(__builtin_bit_cast(float, (uint32_t) r[0]), __builtin_bit_cast(float, (uint32_t) r[1]));
}

typedef __attribute__((address_space(3))) void lds_void_t;

// one LDS-DMA instruction: 64 lanes x 16 bytes, wave-uniform base + per-lane offset -> LDS [lds_byte + lane * 16] (the kernel waits by hand)
__device__ __forceinline__ void dma16(const char* base, uint32_t off, uint32_t lds_byte)
{
    uint32_t m0_keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0" : "=&s"(m0_keep) : "v"(off), "s"(base), "s"(lds_byte) : "memory");
}

// softmax_block over the 16 NN keys of a unit (or of a wave's half of it): score [n][i] of the lane is key key_lane0 + 32 (n / 2) + 4 (n % 2) + i.  `plain`: nothing but a positive
// scale stands between the product and the exponent, which then is one multiply-add and one exponential per score.
template <int VT, int NN>
__device__ __forceinline__ void softmax_unit(f32x4 (&s)[NN], float& m_run, float& l_run, f32x4 (&acc)[VT], uint4 (&pf)[NN / 2], const HeadMods& hm, bool plain,
    bool masked, int key_lane0, int qpos, int klo)
{
    if (!plain)
    {
        // (asked once for all scores: a branch at each one leaves its exponential and its reciprocal to wait for each other, 46 us for 37 at 16 heads of 2 x 64 / 128, 1024 rows)
        auto all = [&](auto&& f) {
#pragma unroll
            for (int n = 0; n < NN; ++n)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    s[n][i] = f(s[n][i], key_lane0 + 32 * (n >> 1) + 4 * (n & 1) + i);
        };
        if (hm.cap2 > 0.f)
            all([&](float v, int) {
                const float t2 = __builtin_amdgcn_exp2f(fminf(fmaxf(v * hm.cap_arg, -43.f), 43.f)); // (softmax_block)
                return hm.cap2 * (t2 - 1.f) * __builtin_amdgcn_rcpf(t2 + 1.f);
            });
        else
            all([&](float v, int) { return v * hm.scale2; });
        if (hm.pen)
        {
            all([&](float v, int key) { return v - hm.slope2 * (float) (qpos - key); });
            if (hm.r1 != 0.f)
                all([&](float v, int key) { return v - hm.r1 * __builtin_amdgcn_logf(fmaxf(1.f + hm.r2 * (float) (qpos - key), 1e-30f)); });
        }
    }
    if (masked)
    {
#pragma unroll
        for (int n = 0; n < NN; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                const int kidx = key_lane0 + 32 * (n >> 1) + 4 * (n & 1) + i;
                if (kidx > qpos || (kidx < klo && kidx >= hm.keep))
                    s[n][i] = -INFINITY;
            }
    }
    if (hm.sigm)
    {
#pragma unroll
        for (int n = 0; n < NN; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                s[n][i] = s[n][i] == -INFINITY ? 0.f : __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-(s[n][i] + hm.wb2)));
    }
    else
    {
        float bm = -INFINITY;
#pragma unroll
        for (int n = 0; n < NN; ++n)
            bm = fmaxf(bm, fmaxf(fmaxf(s[n][0], s[n][1]), fmaxf(s[n][2], s[n][3])));
        const float sc = plain ? hm.scale2 : 1.f;
        const float mn = fmaxf(m_run, rows_max_swap(bm) * sc);
        const bool none = mn == -INFINITY; // this row sees no key of this unit (nor of any before)
        const float corr = none ? 1.f : __builtin_amdgcn_exp2f(m_run - mn), off = none ? 0.f : -mn;
        float rs = 0.f;
#pragma unroll
        for (int n = 0; n < NN; ++n)
        {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                s[n][i] = __builtin_amdgcn_exp2f(fmaf(s[n][i], sc, off));
            rs += (s[n][0] + s[n][1]) + (s[n][2] + s[n][3]);
        }
        l_run = l_run * corr + rs; // (the lane's own keys: the rows' sums meet behind the last unit)
        m_run = mn;
        if (__builtin_amdgcn_ballot_w64(corr != 1.f) != 0) // (softmax_block)
        {
#pragma unroll
            for (int ct = 0; ct < VT; ++ct)
                acc[ct] *= corr;
        }
    }
#pragma unroll
    for (int b = 0; b < NN / 2; ++b)
        pf[b] = make_uint4(pack_bf16(s[2 * b][0], s[2 * b][1]), pack_bf16(s[2 * b][2], s[2 * b][3]), pack_bf16(s[2 * b + 1][0], s[2 * b + 1][1]),
            pack_bf16(s[2 * b + 1][2], s[2 * b + 1][3]));
}

// the bfloat16 infinities and NaNs of x leave it as zeros -> 1.0 in their places
__device__ __forceinline__ uint4 take_specials(uint4& x)
{
    uint32_t v[4] = {x.x, x.y, x.z, x.w}, o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
    {
        const uint32_t top = ((v[i] & 0x7fff7fffu) + 0x00800080u) >> 15 & 0x00010001u; // an exponent of ones carries into the sign's place
        v[i] &= ~(top * 0xffffu);
        o[i] = top * 0x3f80u;
    }
    x = make_uint4(v[0], v[1], v[2], v[3]);
    return make_uint4(o[0], o[1], o[2], o[3]);
}
// 1.0 where a bfloat16 of x is not zero
__device__ __forceinline__ uint4 ones_where(const uint4& x)
{
    const uint32_t v[4] = {x.x, x.y, x.z, x.w};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        o[i] = (v[i] & 0x7fffu ? 0x3f80u : 0u) | (v[i] & 0x7fff0000u ? 0x3f800000u : 0u);
    return make_uint4(o[0], o[1], o[2], o[3]);
}

// attn_prompt_kernel: prompts, heads of 64 / 128 / 192 query and 64 / 128 value dimensions, pages of a multiple of 64 keys.  The products of
// attn_prefill_kernel, with what bounded it taken out (2 us per 32-key block and workgroup, of which the products are 0.1 and the softmax 0.2: the
// staging through registers, two barriers and the shuffles of one block stood one after another):
//   - a unit is 64 keys; its K and V^T rows go to LDS by LDS-DMA, the next unit's in flight under this one's arithmetic (two buffers, ONE barrier per
//     unit); the 16-byte pieces of a row are permuted at the source so that the fragment reads fall on different banks;
//   - a wave owns RT tiles of 16 rows (a workgroup 64 RT rows): every fragment read from LDS feeds all of them;
//   - tile t of a half unit holds keys 8 (r / 4) + 4 t + r % 4 in row r, so that a lane's eight scores are eight neighbouring keys and the V^T fragment
//     that meets them is one 16-byte read;
//   - a row's maximum meets over the lanes by register swaps;
//   - KS = 2 (few workgroups): two waves to a row tile, each with its half of every unit's keys, a workgroup 32 rows; they meet behind the last unit.
// Workgroups: the heaviest tiles of all heads first, the heads of one key/value head on one XCD.  Up to two to a CU, workgroup i + CUs shares i's: from tile level `turn` on the lightest
// come first, so that a CU has 17 units of a prompt's 32 rows, and not 24 or 9.
// Measured (us): 32 heads over 8, 192 / 128, 2048 rows at contexts 0 and 2048 on average 402 -> 149, without waits for the next unit inside the walk 127; 128 / 128 272 -> 133 -> 114; 16
// heads of 2 x 64 / 128 with a soft cap, 1024 rows 90 -> 53, with workgroups of 32 rows for 64, on eight waves, and the turn 46, with the soft cap's branch asked once a unit (softmax_unit)
// 37, without those waits 34.
template <int MAPS, int DK, int VT, int RT, int KS>
__global__ __launch_bounds__(256, 2) void attn_prompt_kernel(const StackAttnParams p, int min_count, int tiles, int turn)
{
    constexpr int RW = 4 / KS, D = DK * 32, V = VT * 16, ROWS = 16 * RW * RT; // RW: waves of different rows
    constexpr int KPR = D / 8;                                    // 16-byte pieces of a K row
    constexpr int NW = 4, NN = 4 / KS;                            // waves; score tiles of 16 keys per wave and unit
    constexpr int KI = MAPS * KPR / NW, VI = V / 8 / NW;          // DMA instructions per wave and unit
    constexpr int KB = MAPS * 64 * D * 2, BUF = KB + V * 128;     // bytes
    // Fragments read ahead of their products (V's: over the softmax), what 256 registers have room for: left to itself the compiler waits for each pair of them, LDS answers in 100 clocks
    // and the products of one take 32 (us, 32 heads, 2048 rows at contexts 0 and 2048 on average: 192 / 128 127 -> 118, 128 / 128 114 -> 106).
    constexpr int AHEAD = RT * DK > 8 ? 3 : 4, V_AHEAD = RT * DK > 8 ? 2 : 4;
    static_assert(KPR % 8 == 0 && V % 64 == 0 && MAPS * KPR % NW == 0, "head sizes");
    extern __shared__ __attribute__((aligned(16))) char smem[];
    // blockIdx.x = tile level x (entries x heads), heaviest tiles first; inside a level the key/value heads run fastest
    const int per = p.entries * p.heads;
    const int level = prompt_level(blockIdx.x / per, turn, tiles), q_ = blockIdx.x % per, e = q_ / p.heads, hi = q_ % p.heads;
    const int h = p.cross_values ? hi : hi % p.kv_heads * (p.heads / p.kv_heads) + hi / p.kv_heads;
    const int count = p.ent_count[e];
    if (count < min_count)
        return;
    const int tile = (count + ROWS - 1) / ROWS - 1 - level;
    if (tile < 0)
        return;
    const int first = p.ent_first[e], pos0 = p.ent_pos0[e];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, g4 = lane >> 4, wr = w % RW, half = w / RW; // row tile, and which half of a unit's keys (KS = 2)
    const HeadMap hd = head_map(p, h);
    const int page = p.page, upp = page / 64; // units per page
    const int32_t* table = p.block_table + (int64_t) e * p.max_blocks;
    const HeadMods hm = head_mods(p, h);
    const bool plain = hm.cap2 == 0.f && !hm.pen && !hm.sigm && hm.scale2 > 0.f;

    int r0[RT], qpos[RT], klo[RT], my_last[RT], my_lo[RT], klo_last[RT];
    bf16x8 qf[RT][MAPS][DK];
    float m_run[RT][MAPS], l_run[RT][MAPS];
    f32x4 acc[RT][MAPS][VT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
    {
        r0[rt] = tile * ROWS + (wr * RT + rt) * 16;
        const bool rows_ok = r0[rt] < count; // wave-uniform
        const int qrow = r0[rt] + col < count ? r0[rt] + col : count - 1;
        qpos[rt] = pos0 + qrow;
        klo[rt] = first_visible(p, qpos[rt]);
#pragma unroll
        for (int m = 0; m < MAPS; ++m)
        {
#pragma unroll
            for (int ks = 0; ks < DK; ++ks)
                qf[rt][m][ks] = as_bf16x8(*reinterpret_cast<const uint4*>(
                    reinterpret_cast<const uint16_t*>(p.q) + (((int64_t) (first + qrow) * hd.q_heads + hd.qh) * MAPS + m) * D + ks * 32 + 8 * g4));
        }
        const int last = r0[rt] + 15 < count ? r0[rt] + 15 : count - 1;
        my_last[rt] = rows_ok ? (pos0 + last) / 64 : -1; // the tile's last unit that holds a visible key, and its first
        my_lo[rt] = rows_ok ? first_visible(p, pos0 + r0[rt]) / 64 : 0;
        klo_last[rt] = rows_ok ? first_visible(p, pos0 + last) : 0;
    }
    const int wg_last = tile * ROWS + ROWS - 1 < count ? tile * ROWS + ROWS - 1 : count - 1;
    // the units the workgroup walks: the ones with kept first keys, then from its first row's first visible key on
    const int lo = first_visible(p, pos0 + tile * ROWS) / 64;
    const int keep_u = (p.mask == MASK_WINDOW && p.mask_keep > 0) ? (p.mask_keep + 63) / 64 : 0, nkeep = keep_u < lo ? keep_u : lo;
    const int n_units = nkeep + (pos0 + wg_last) / 64 + 1 - lo;
    auto unit_at = [&](int v) { return v < nkeep ? v : v - nkeep + lo; };

    // this lane's part of a unit's DMA: instruction i of wave w fills LDS pieces (NW i + w) 64 + lane
    uint32_t koff[KI], voff[VI];
#pragma unroll
    for (int i = 0; i < KI; ++i)
    {
        const int L = (i * NW + w) * 64 + lane, row = L / KPR, pc = L % KPR, r = row % 64;
        const int x = KPR % 16 == 0 ? ((r >> 3) & 3) << 2 | (r & 3) : ((r >> 3) & 3) << 1 | ((r >> 1) & 1);
        koff[i] = (uint32_t) ((row / 64 * page + r) * D * 2 + (pc ^ x) * 16);
    }
#pragma unroll
    for (int i = 0; i < VI; ++i)
    {
        const int L = (i * NW + w) * 64 + lane, row = L / 8, pc = L % 8;
        voff[i] = (uint32_t) (row * page * 2 + (pc ^ ((row >> 1) & 7)) * 16);
    }
    const uint32_t lds0 = (uint32_t) (uintptr_t) (lds_void_t*) smem + w * 1024;
    auto request = [&](int u, int blk, int buf) {
        const int off = upp == 1 ? 0 : u % upp * 64;
        const char* kb = reinterpret_cast<const char*>(p.k_pool) + (((int64_t) blk * (p.kv_heads * MAPS) + hd.kh * MAPS) * page + off) * D * 2;
        const char* vb = reinterpret_cast<const char*>(p.v_pool) + (((int64_t) blk * p.kv_heads + hd.vh) * V * page + off) * 2;
#pragma unroll
        for (int i = 0; i < KI; ++i)
            dma16(kb, koff[i], lds0 + buf * BUF + i * NW * 1024);
#pragma unroll
        for (int i = 0; i < VI; ++i)
            dma16(vb, voff[i], lds0 + buf * BUF + KB + i * NW * 1024);
    };
    auto block_of = [&](int u) { return table[upp == 1 ? u : u / upp]; };

    // CAREFUL: a value that is no finite number meets only the rows that see its key (a weight of 0 times it would make it everyone's)
    auto walk = [&](auto careful) {
        constexpr bool CAREFUL = decltype(careful)::value;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int m = 0; m < MAPS; ++m)
            {
                m_run[rt][m] = -INFINITY;
                l_run[rt][m] = 0.f;
#pragma unroll
                for (int ct = 0; ct < VT; ++ct)
                    acc[rt][m][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        request(unit_at(0), __builtin_amdgcn_readfirstlane(block_of(unit_at(0))), 0);
        // (in a vector register until behind the next unit's wait: earlier, its own would be one for the requests in front of it)
        int blk_next = n_units > 1 ? block_of(unit_at(1)) : 0;
        // The queries' fragments are here: a wait for them inside the loop, where the compiler would leave it, is one for the next unit's K and V, too (they are requested in front of it).
        // Ahead of the first request, their way and the page number's and K's and V's would follow each other: 2.4 % over 1274 steps of up to 8 prompts and 4096 rows, 3 - 7 % of short ones (45 of
        // those steps took over 1.03 of the time without any such wait; 4 do so, up to 1.05).
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int m = 0; m < MAPS; ++m)
#pragma unroll
                for (int ks = 0; ks < DK; ++ks)
                    asm volatile("" : "+v"(qf[rt][m][ks]));
        for (int v = 0; v < n_units; ++v)
        {
            const int u = unit_at(v);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads(); // the unit has landed for every wave, and every wave is through with the one before it
            if (v + 1 < n_units)
            {
                request(unit_at(v + 1), __builtin_amdgcn_readfirstlane(blk_next), (v + 1) & 1);
                if (v + 2 < n_units)
                    blk_next = block_of(unit_at(v + 2));
            }
            bool on[RT], any = false; // wave-uniform
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
            {
                on[rt] = u <= my_last[rt] && (u >= my_lo[rt] || u < keep_u);
                any = any || on[rt];
            }
            if (!any)
                continue;
            const char* ks_ = smem + (v & 1) * BUF;
            const char* vs_ = ks_ + KB;
            const int key0 = u * 64 + (KS == 2 ? half * 32 : 0);
            uint4 pf[RT][MAPS][NN / 2], vf[VT * NN / 2];
            auto v_at = [&](int x) {
                const int row = x / (NN / 2) * 16 + col, b = x % (NN / 2);
                return *reinterpret_cast<const uint4*>(vs_ + row * 128 + ((((KS == 2 ? half : b) * 4 + g4) ^ ((row >> 1) & 7)) << 4));
            };
#pragma unroll
            for (int m = 0; m < MAPS; ++m)
            {
                f32x4 s[RT][NN];
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                    for (int n = 0; n < NN; ++n)
                        s[rt][n] = f32x4{0.f, 0.f, 0.f, 0.f};
                // fragments of two score tiles in turn
                auto k_at = [&](int x) {
                    const int n = x / (2 * DK) * 2 + x % 2, ks = x / 2 % DK;
                    const int r = 32 * (KS == 2 ? half : n >> 1) + 8 * (col >> 2) + 4 * (n & 1) + (col & 3);
                    const int sw = KPR % 16 == 0 ? ((r >> 3) & 3) << 2 | (r & 3) : ((r >> 3) & 3) << 1 | ((r >> 1) & 1);
                    return *reinterpret_cast<const uint4*>(ks_ + (m * 64 + r) * (D * 2) + (((ks * 4 + g4) ^ sw) << 4));
                };
                uint4 kf[NN * DK];
#pragma unroll
                for (int x = 0; x < AHEAD; ++x)
                    kf[x] = k_at(x);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int x = 0; x < NN * DK; ++x)
                {
                    const int n = x / (2 * DK) * 2 + x % 2, ks = x / 2 % DK;
                    if (x + AHEAD < NN * DK)
                        kf[x + AHEAD] = k_at(x + AHEAD);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt) // (no branches among the products: a tile that is off has its scores dropped below)
                        s[rt][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(kf[x]), qf[rt][m][ks], s[rt][n], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (m == MAPS - 1)
                {
#pragma unroll
                    for (int x = 0; x < V_AHEAD; ++x)
                        vf[x] = v_at(x);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
                {
                    pf[rt][m][0] = pf[rt][m][NN / 2 - 1] = make_uint4(0, 0, 0, 0);
                    if (RT == 1 || on[rt])
                    {
                        const bool masked = key0 + 16 * NN - 1 > pos0 + r0[rt] || key0 < klo_last[rt];
                        softmax_unit<VT, NN>(s[rt], m_run[rt][m], l_run[rt][m], acc[rt][m], pf[rt][m], hm, plain, masked, key0 + 8 * g4, qpos[rt], klo[rt]);
                    }
                }
            }
#pragma unroll
            for (int ct = 0; ct < VT; ++ct)
#pragma unroll
                for (int b = 0; b < NN / 2; ++b)
                {
                    constexpr int ALL = VT * NN / 2;
                    const int x = ct * (NN / 2) + b;
                    if (x + V_AHEAD < ALL)
                        vf[x + V_AHEAD] = v_at(x + V_AHEAD);
                    __builtin_amdgcn_sched_barrier(0);
                    uint4 vr = vf[x];
                    uint4 vbad = make_uint4(0, 0, 0, 0);
                    if constexpr (CAREFUL)
                        vbad = take_specials(vr);
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                        for (int m = 0; m < MAPS; ++m)
                        {
                            acc[rt][m][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(vr), as_bf16x8(pf[rt][m][b]), acc[rt][m][ct], 0, 0, 0);
                            if constexpr (CAREFUL)
                            {
                                const f32x4 n = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(vbad), as_bf16x8(ones_where(pf[rt][m][b])), f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                                for (int i = 0; i < 4; ++i)
                                    acc[rt][m][ct][i] = n[i] > 0.f ? __builtin_nanf("") : acc[rt][m][ct][i];
                            }
                        }
                    __builtin_amdgcn_sched_barrier(0);
                }
        }
    };
    walk(std::false_type());
    {
        // A row that is not finite, in any wave: once more, carefully.  (Asked once, behind the last unit.)
        bool finite = true;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int m = 0; m < MAPS; ++m)
#pragma unroll
                for (int ct = 0; ct < VT; ++ct)
                    finite = finite && (fabsf(acc[rt][m][ct][0]) + fabsf(acc[rt][m][ct][1])) + (fabsf(acc[rt][m][ct][2]) + fabsf(acc[rt][m][ct][3])) < INFINITY;
        int* flags = reinterpret_cast<int*>(smem);
        const bool mine = __builtin_amdgcn_ballot_w64(!finite) != 0;
        __syncthreads(); // (the waves are through with the last unit)
        if (lane == 0)
            flags[w] = mine ? 1 : 0;
        __syncthreads();
        int any = 0;
#pragma unroll
        for (int i = 0; i < NW; ++i)
            any |= flags[i];
        if (__builtin_amdgcn_readfirstlane(any))
        {
            __syncthreads(); // (the flags' place is the first unit's)
            walk(std::true_type());
        }
    }
    if constexpr (KS == 2)
    {
        // the two halves of the keys meet: waves RW .. 2 RW - 1 leave theirs in LDS
        static_assert(RT == 1, "one row tile per wave");
        constexpr int PER = (VT * 4 + 2) * 64; // floats per wave and map
        float* x = reinterpret_cast<float*>(smem) + wr * PER * MAPS + lane;
        __syncthreads();
        if (half)
        {
#pragma unroll
            for (int m = 0; m < MAPS; ++m)
            {
                x[m * PER] = m_run[0][m];
                x[m * PER + 64] = l_run[0][m];
#pragma unroll
                for (int ct = 0; ct < VT; ++ct)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        x[m * PER + (2 + ct * 4 + i) * 64] = acc[0][m][ct][i];
            }
        }
        __syncthreads();
        if (half)
            return;
#pragma unroll
        for (int m = 0; m < MAPS; ++m)
        {
            const float m1 = x[m * PER], M = fmaxf(m_run[0][m], m1);
            const float f0 = hm.sigm ? 1.f : (m_run[0][m] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run[0][m] - M));
            const float f1 = hm.sigm ? 1.f : (m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m1 - M));
            m_run[0][m] = M;
            l_run[0][m] = l_run[0][m] * f0 + x[m * PER + 64] * f1;
#pragma unroll
            for (int ct = 0; ct < VT; ++ct)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    acc[0][m][ct][i] = acc[0][m][ct][i] * f0 + x[m * PER + (2 + ct * 4 + i) * 64] * f1;
        }
    }
    // lane (col, g4) holds, for row col of a tile, channels ct * 16 + 4 g4 + i
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
    {
        float inv[MAPS];
#pragma unroll
        for (int m = 0; m < MAPS; ++m)
            inv[m] = finish_factor(p, h, m_run[rt][m], rows_sum(l_run[rt][m]));
        float ss = 0.f;
#pragma unroll
        for (int ct = 0; ct < VT; ++ct)
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                float o = acc[rt][0][ct][i] * inv[0];
                if (MAPS == 2)
                    o -= p.lambda * (acc[rt][MAPS - 1][ct][i] * inv[MAPS - 1]);
                acc[rt][0][ct][i] = o;
                ss += o * o;
            }
        float mul = 1.f;
        if (p.head_norm)
            mul = p.out_scale / sqrtf(rows_sum(ss) / (float) V + p.eps);
        if (r0[rt] + col < count)
        {
            mul *= out_gate_of(p, first + r0[rt] + col, h);
            uint16_t* out = reinterpret_cast<uint16_t*>(p.out) + ((int64_t) (first + r0[rt] + col) * p.heads + h) * V + 4 * g4;
#pragma unroll
            for (int ct = 0; ct < VT; ++ct)
                *reinterpret_cast<uint2*>(out + ct * 16) = make_uint2(pack_bf16(acc[rt][0][ct][0] * mul, acc[rt][0][ct][1] * mul),
                    pack_bf16(acc[rt][0][ct][2] * mul, acc[rt][0][ct][3] * mul));
        }
    }
}

template <int MAPS, int DK, int VT, int RT, int KS>
void launch_prompt(const StackAttnParams& p, int min_count, hipStream_t stream)
{
    constexpr int RW = 4 / KS;
    constexpr size_t stages = 2 * ((size_t) MAPS * 64 * DK * 64 + VT * 16 * 128), merge = KS == 2 ? (size_t) RW * MAPS * (VT * 4 + 2) * 256 : 0;
    constexpr size_t lds = stages > merge ? stages : merge;
    launch_util::ensure_dynamic_lds(reinterpret_cast<const void*>(&attn_prompt_kernel<MAPS, DK, VT, RT, KS>), lds);
    const int tiles = (p.max_count + 16 * RW * RT - 1) / (16 * RW * RT);
    const int64_t per = (int64_t) p.entries * p.heads;
    const int turn = prompt_turn(tiles, per, launch_util::device_cus());
    hipLaunchKernelGGL((attn_prompt_kernel<MAPS, DK, VT, RT, KS>), dim3((unsigned) (tiles * per)), dim3(256), lds, stream, p, min_count, tiles, turn);
}

// attn_prefill_wide_kernel: the staged form for one map and long rows (dim of 160 and more), where the fragment reads out of LDS, not
// the matrix pipe, bound attn_prefill_kernel: a wave owns TWO 16-row tiles (a workgroup 128 rows) and every K and V^T fragment it reads
// from LDS feeds both, which halves the LDS traffic per score.  Same staging, same products, same finish.
template <int DK, int VT>
__global__ __launch_bounds__(256) void attn_prefill_wide_kernel(const StackAttnParams p, int min_count)
{
    constexpr int RT = 2, ROWS = 64 * RT;
    constexpr int D = DK * 32, V = VT * 16;
    constexpr int KP = D * 2 + 16, VP = 80;
    constexpr int K16 = 32 * (D / 8), V16 = V * 4;
    constexpr int KPT = (K16 + 255) / 256, VPT = (V16 + 255) / 256;
    __shared__ __attribute__((aligned(16))) char k_s[32 * KP];
    __shared__ __attribute__((aligned(16))) char v_s[V * VP];
    const int e = blockIdx.y, h = blockIdx.z;
    const int count = p.ent_count[e];
    if (count < min_count)
        return;
    const int tile = (count + ROWS - 1) / ROWS - 1 - (int) blockIdx.x;
    if (tile < 0)
        return;
    const int first = p.ent_first[e], pos0 = p.ent_pos0[e];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int col = lane & 15, g4 = lane >> 4;
    const HeadMap hd = head_map(p, h);
    const int g = hd.kh, gv = hd.vh;
    const int page = p.page;
    const int32_t* table = p.block_table + (int64_t) e * p.max_blocks;
    const HeadMods hm = head_mods(p, h);
    const uint16_t* kp = reinterpret_cast<const uint16_t*>(p.k_pool);
    const uint16_t* vp = reinterpret_cast<const uint16_t*>(p.v_pool);

    int r0[RT], qpos[RT], klo[RT], my_blk[RT], my_lo[RT], klo_last[RT];
    bool rows_ok[RT];
    bf16x8 qf[RT][DK];
    float m_run[RT], l_run[RT];
    f32x4 acc[RT][VT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
    {
        r0[rt] = tile * ROWS + (w * RT + rt) * 16;
        rows_ok[rt] = r0[rt] < count; // wave-uniform
        const int qrow = r0[rt] + col < count ? r0[rt] + col : count - 1;
        qpos[rt] = pos0 + qrow;
        klo[rt] = first_visible(p, qpos[rt]);
#pragma unroll
        for (int ks = 0; ks < DK; ++ks)
            qf[rt][ks] = as_bf16x8(*reinterpret_cast<const uint4*>(
                reinterpret_cast<const uint16_t*>(p.q) + ((int64_t) (first + qrow) * hd.q_heads + hd.qh) * D + ks * 32 + 8 * g4));
        const int my_last = r0[rt] + 15 < count ? r0[rt] + 15 : count - 1;
        my_blk[rt] = rows_ok[rt] ? (pos0 + my_last) / 32 : -1;
        my_lo[rt] = rows_ok[rt] ? first_visible(p, pos0 + r0[rt]) / 32 : 0;
        klo_last[rt] = rows_ok[rt] ? first_visible(p, pos0 + my_last) : 0;
        m_run[rt] = -INFINITY;
        l_run[rt] = 0.f;
#pragma unroll
        for (int ct = 0; ct < VT; ++ct)
            acc[rt][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const int wg_last = tile * ROWS + ROWS - 1 < count ? tile * ROWS + ROWS - 1 : count - 1;
    const int nblk = (pos0 + wg_last) / 32 + 1;
    const int wg_lo = first_visible(p, pos0 + tile * ROWS) / 32;

    u32x4 kr[KPT], vr[VPT];
    const BlockWalk bw = block_walk(p, pos0 + tile * ROWS, nblk);
    // blocks below this index hold kept first keys, which every row sees whatever its own window (a wave whose rows start further
    // down than the workgroup's first takes part in them too)
    const int keep_blk = (p.mask == MASK_WINDOW && p.mask_keep > 0) ? (p.mask_keep + 31) / 32 : 0;
    int blk_next = table[walk_block(bw, 0) * 32 / page];
    auto request = [&](int vb) {
        const int key0 = walk_block(bw, vb) * 32;
        const int blk = blk_next, off = key0 % page;
        blk_next = table[vb + 1 < bw.n ? walk_block(bw, vb + 1) * 32 / page : key0 / page];
#pragma unroll
        for (int i = 0; i < KPT; ++i)
        {
            const int idx = tid + i * 256;
            if (K16 % 256 == 0 || idx < K16)
            {
                const int row = idx / (D / 8), piece = idx % (D / 8);
                kr[i] = *reinterpret_cast<const u32x4*>(kp + (((int64_t) blk * p.kv_heads + g) * page + off + row) * D + piece * 8);
            }
        }
#pragma unroll
        for (int i = 0; i < VPT; ++i)
        {
            const int idx = tid + i * 256;
            if (V16 % 256 == 0 || idx < V16)
                vr[i] = *reinterpret_cast<const u32x4*>(vp + (((int64_t) blk * p.kv_heads + gv) * V + idx / 4) * page + off + (idx % 4) * 8);
        }
    };
    request(0);
    for (int vb = 0; vb < bw.n; ++vb)
    {
        const int kb = walk_block(bw, vb);
#pragma unroll
        for (int i = 0; i < KPT; ++i)
        {
            const int idx = tid + i * 256;
            if (K16 % 256 == 0 || idx < K16)
                *reinterpret_cast<u32x4*>(k_s + (idx / (D / 8)) * KP + (idx % (D / 8)) * 16) = kr[i];
        }
#pragma unroll
        for (int i = 0; i < VPT; ++i)
        {
            const int idx = tid + i * 256;
            if (V16 % 256 == 0 || idx < V16)
                *reinterpret_cast<u32x4*>(v_s + (idx / 4) * VP + (idx % 4) * 16) = vr[i];
        }
        __syncthreads();
        if (vb + 1 < bw.n)
            request(vb + 1);
        bool on[RT]; // wave-uniform
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
            on[rt] = kb <= my_blk[rt] && (kb >= my_lo[rt] || kb < keep_blk);
        if (on[0] || on[RT - 1])
        {
            const int key0 = kb * 32;
            f32x4 s[RT][2];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
                s[rt][0] = s[rt][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int ks = 0; ks < DK; ++ks)
                {
                    const bf16x8 kfr = as_bf16x8(*reinterpret_cast<const uint4*>(k_s + (t * 16 + col) * KP + (ks * 32 + 8 * g4) * 2));
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt) // (no branches among the products: a tile that is off has its scores dropped below)
                        s[rt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kfr, qf[rt][ks], s[rt][t], 0, 0, 0);
                }
            uint4 pf[RT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
            {
                pf[rt] = make_uint4(0, 0, 0, 0);
                if (on[rt])
                {
                    const bool masked = key0 + 31 > pos0 + r0[rt] || key0 < klo_last[rt];
                    pf[rt] = softmax_block<VT>(s[rt], m_run[rt], l_run[rt], acc[rt], hm, masked, key0 + 4 * g4, qpos[rt], klo[rt]);
                }
            }
#pragma unroll
            for (int ct = 0; ct < VT; ++ct)
            {
                const char* vrow = v_s + (ct * 16 + col) * VP + 8 * g4;
                const uint2 lo = *reinterpret_cast<const uint2*>(vrow);
                const uint2 hi = *reinterpret_cast<const uint2*>(vrow + 32);
                const bf16x8 vf = as_bf16x8(make_uint4(lo.x, lo.y, hi.x, hi.y));
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
                    acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, as_bf16x8(pf[rt]), acc[rt][ct], 0, 0, 0);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
    {
        const float l_sum = rows_sum(l_run[rt]);
        if (!rows_ok[rt] || r0[rt] + col >= count)
            continue;
        const float mul = finish_factor(p, h, m_run[rt], l_sum) * out_gate_of(p, first + r0[rt] + col, h);
        uint16_t* out = reinterpret_cast<uint16_t*>(p.out) + ((int64_t) (first + r0[rt] + col) * p.heads + h) * V + 4 * g4;
#pragma unroll
        for (int ct = 0; ct < VT; ++ct)
            *reinterpret_cast<uint2*>(out + ct * 16)
                = make_uint2((uint32_t) f2bf(acc[rt][ct][0] * mul) | ((uint32_t) f2bf(acc[rt][ct][1] * mul) << 16),
                    (uint32_t) f2bf(acc[rt][ct][2] * mul) | ((uint32_t) f2bf(acc[rt][ct][3] * mul) << 16));
    }
}

// Second pass of the key split: one wave per (row, head) combines the ks partials of each map, then the differential combination,
// the head norm and the bfloat16 store.
template <int MAPS>
__global__ __launch_bounds__(64) void attn_split_merge_kernel(const StackAttnParams p, int ks, int below_count)
{
    const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
    if (p.ent_count[p.tok_entry[t]] >= below_count)
        return;
    const int V = p.vdim;
    const float* base = p.split_ws + (((int64_t) t * p.heads + h) * ks) * MAPS * (V + 2);
    // lane l < ks * MAPS owns partial (split l / MAPS, map l % MAPS): all maxima and sums are fetched at once, the weights are
    // formed with wave reductions and handed to the channel lanes by shuffles
    const bool owner = lane < ks * MAPS;
    const float pm = owner ? base[lane * (V + 2) + V] : -INFINITY;
    const float pl = owner ? base[lane * (V + 2) + V + 1] : 0.f;
    float wl = 0.f;
#pragma unroll
    for (int m = 0; m < MAPS; ++m)
    {
        const bool mine = owner && lane % MAPS == m;
        const float M = wave_max(mine ? pm : -INFINITY);
        const float e_ = p.weights == WEIGHTS_SIGMOID ? 1.f : (mine && pm != -INFINITY ? __builtin_amdgcn_exp2f(pm - M) : 0.f);
        const float L = wave_sum(mine ? e_ * pl : 0.f);
        if (mine)
            wl = e_ * finish_factor(p, h, M, L);
    }
    constexpr int MC = 4; // vdim <= 256: four channels per lane
    float o[MC], ss = 0.f;
    float a[MC][MAPS];
#pragma unroll
    for (int c = 0; c < MC; ++c)
#pragma unroll
        for (int m = 0; m < MAPS; ++m)
            a[c][m] = 0.f;
    // four partials at a time, every load of them requested before the first is used (partials beyond the last: the last again, weight 0)
    const int n_part = ks * MAPS;
    for (int i0 = 0; i0 < n_part; i0 += 4)
    {
        float v[4][MC];
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            const float* part = base + (int64_t) (i0 + j < n_part ? i0 + j : n_part - 1) * (V + 2);
#pragma unroll
            for (int c = 0; c < MC; ++c)
                v[j][c] = part[lane + c * 64 < V ? lane + c * 64 : V - 1];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            const float wgt = i0 + j < n_part ? __shfl(wl, i0 + j, 64) : 0.f;
#pragma unroll
            for (int c = 0; c < MC; ++c)
                a[c][j % MAPS] += wgt * v[j][c]; // (i0 is a multiple of 4: partial i0 + j belongs to map j % MAPS)
        }
    }
#pragma unroll
    for (int c = 0; c < MC; ++c)
    {
        o[c] = 0.f;
        if (lane + c * 64 < V)
        {
            o[c] = MAPS == 2 ? a[c][0] - p.lambda * a[c][MAPS - 1] : a[c][0];
            ss += o[c] * o[c];
        }
    }
    float mul = 1.f;
    if (p.head_norm)
        mul = p.out_scale / sqrtf(wave_sum(ss) / (float) V + p.eps);
    mul *= out_gate_of(p, t, h);
    uint16_t* out = reinterpret_cast<uint16_t*>(p.out) + ((int64_t) t * p.heads + h) * V;
#pragma unroll
    for (int c = 0; c < MC; ++c)
        if (lane + c * 64 < V)
            out[lane + c * 64] = f2bf(o[c] * mul);
}

template <int MAPS, int DK, int VT>
int launch_tile(const StackAttnParams& p, hipStream_t stream)
{
    constexpr int NW = 4;
    const size_t lds = sizeof(float) * ((size_t) NW * MAPS * 16 * (VT * 16 + 16) + (size_t) NW * MAPS * 16 * 2);
    // entries of PREFILL_ROWS rows and more go to the staged form, the rest (decoded tokens, short portions) to the key-split form;
    // a mixed step launches both, each skipping the other's entries
    static const int PREFILL_ROWS = [] {
        const char* v = std::getenv("TLLM_STACK_PREFILL_ROWS"); // measurement knob: rows from which an entry takes the staged form
        return v && std::atoi(v) > 0 ? std::atoi(v) : 32;
    }();
    const int small_rows = p.max_count < PREFILL_ROWS ? p.max_count : (p.tokens > p.max_count ? PREFILL_ROWS - 1 : 0);
    if (p.max_count >= PREFILL_ROWS)
    {
        // the wide form (128 rows per workgroup) where it still fills the chip; otherwise twice as many workgroups of 64 rows
        bool wide = false;
        if constexpr (MAPS == 1 && DK >= 5)
        {
            const char* force = std::getenv("TLLM_STACK_WIDE_PREFILL"); // test / measurement knob: 1 = always, 0 = never
            // (shapes whose 64-row form fits two waves per SIMD run that one: twice the waves hide what the wide form saves in LDS reads)
            wide = !p.head_norm
                && (force ? force[0] == '1' : DK >= 10 && (int64_t) ((p.max_count + 127) / 128) * p.entries * p.heads >= launch_util::device_cus());
        }
        if constexpr (MAPS == 1 && DK >= 5)
        {
            if (wide)
            {
                const dim3 pg((p.max_count + 127) / 128, p.entries, p.heads);
                hipLaunchKernelGGL((attn_prefill_wide_kernel<DK, VT>), pg, dim3(256), 0, stream, p, PREFILL_ROWS);
            }
        }
        // heads of the usual sizes over pages of whole 64-key units (16-byte DMA from both pools); its grid is one-dimensional, and a grid
        // dimension holds fewer than 2^32 threads
        constexpr bool prompt_form = (DK == 2 || DK == 4 || (DK == 6 && MAPS == 1)) && (VT == 4 || VT == 8);
        bool prompt = false;
        if constexpr (prompt_form)
        {
            prompt = p.page % 64 == 0 && !(reinterpret_cast<uintptr_t>(p.v_pool) & 15) && !wide
                && (int64_t) ((p.max_count + 63) / 64) * p.entries * p.heads < (1 << 24);
            if (prompt)
            {
                // two row tiles per wave where such workgroups still make two per CU; waves that share a unit's keys where workgroups of 64 rows
                // would leave one wave to a SIMD
                const int64_t wgs = (int64_t) ((p.max_count + 63) / 64) * p.entries * p.heads, cus = launch_util::device_cus();
                bool two = false;
                if constexpr (MAPS == 1)
                {
                    two = (int64_t) ((p.max_count + 127) / 128) * p.entries * p.heads >= 2 * cus;
                    if (two)
                        launch_prompt<MAPS, DK, VT, 2, 1>(p, PREFILL_ROWS, stream);
                }
                if (two)
                    ;
                else if (wgs <= cus)
                    launch_prompt<MAPS, DK, VT, 1, 2>(p, PREFILL_ROWS, stream);
                else
                    launch_prompt<MAPS, DK, VT, 1, 1>(p, PREFILL_ROWS, stream);
            }
        }
        if (!wide && !prompt)
        {
            const dim3 pg((p.max_count + 63) / 64, p.entries, p.heads);
            hipLaunchKernelGGL((attn_prefill_kernel<MAPS, DK, VT>), pg, dim3(256), 0, stream, p, PREFILL_ROWS);
        }
    }
    if (small_rows > 0)
    {
        // a step of decoded tokens only (every entry within one tile, few rows in all): the keys of an (entry, head) are split over
        // ks workgroups so that a long context is walked by ks * NW waves, two key blocks or so each
        // single decoded tokens whose heads share key/value heads and carry no per-head score numbers: up to 16 heads of a group are the
        // tile's rows (a sink or an output gate is looked up per row)
        const int head_rows = (p.max_count == 1 && p.heads / p.kv_heads >= 4 && !p.cross_values && MAPS == 1 && !p.temp && !p.slope && !p.log_r1
                                  && !p.wbias && !p.head_norm)
            ? (p.heads / p.kv_heads + 15) / 16
            : 0;
        const int gz = head_rows ? p.kv_heads * head_rows : p.heads;
        int ks = 1;
        if (p.split_ws && p.max_count <= 16 && p.tokens <= kSplitRows)
        {
            // a window or a chunk bounds the keys a row walks
            const int span = p.mask == MASK_CAUSAL ? p.max_context
                                                   : std::min(p.max_context, p.mask_size + 31 + (p.mask_keep > 0 ? p.mask_keep + 31 : 0));
            const int nblk = (span + 31) / 32;
            // two key blocks per wave, or one where that still leaves CUs without work
            ks = std::min(kMaxSplits, (nblk + 2 * NW - 1) / (2 * NW));
            if (ks * p.entries * gz * 2 <= launch_util::device_cus())
                ks = std::min(kMaxSplits, (nblk + NW - 1) / NW);
        }
        const dim3 grid(ks > 1 ? ks : (small_rows + 15) / 16, p.entries, gz);
        const auto tile = ks > 1 ? attn_tile_kernel<MAPS, DK, VT, NW, true> : attn_tile_kernel<MAPS, DK, VT, NW, false>;
        launch_util::ensure_dynamic_lds(reinterpret_cast<const void*>(tile), lds);
        hipLaunchKernelGGL(tile, grid, dim3(NW * 64), lds, stream, p, PREFILL_ROWS, ks, head_rows);
        if (ks > 1)
            hipLaunchKernelGGL((attn_split_merge_kernel<MAPS>), dim3(p.tokens, p.heads), dim3(64), 0, stream, p, ks, PREFILL_ROWS);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
    {
        set_error("stack_attention (tile kernels) launch failed: %s", hipGetErrorString(e));
        return -1;
    }
    return 0;
}

template <int MAPS, int DK>
int launch_tile_v(const StackAttnParams& p, hipStream_t stream)
{
    switch (p.vdim)
    {
    case 32: return launch_tile<MAPS, DK, 2>(p, stream);
    case 64: return launch_tile<MAPS, DK, 4>(p, stream);
    case 128: return launch_tile<MAPS, DK, 8>(p, stream);
    }
    if constexpr (MAPS == 1)
        if (p.vdim == 96)
            return launch_tile<MAPS, DK, 6>(p, stream);
    return 1;
}

// one shared key/value head of dim = latent + rotated part, vdim = latent (latent attention in absorbed form)
int launch_tile_latent(const StackAttnParams& p, hipStream_t stream)
{
    if (p.dim == 160 && p.vdim == 128)
        return launch_tile<1, 5, 8>(p, stream);
    if (p.dim == 320 && p.vdim == 256)
        return launch_tile<1, 10, 16>(p, stream);
    // no rotated part: the key row is the latent alone (32 to 128 are the ordinary shapes)
    if (p.dim == p.vdim)
        switch (p.dim)
        {
        case 192: return launch_tile<1, 6, 12>(p, stream);
        case 256: return launch_tile<1, 8, 16>(p, stream);
        }
    return 1;
}

template <int MAPS>
int launch_tile_d(const StackAttnParams& p, hipStream_t stream)
{
    switch (p.dim)
    {
    case 32: return launch_tile_v<MAPS, 1>(p, stream);
    case 64: return launch_tile_v<MAPS, 2>(p, stream);
    case 128: return launch_tile_v<MAPS, 4>(p, stream);
    }
    if constexpr (MAPS == 1)
        switch (p.dim)
        {
        case 96: return launch_tile_v<MAPS, 3>(p, stream);
        case 192: return launch_tile_v<MAPS, 6>(p, stream);
        }
    return 1;
}

} // namespace

// partials of the cross-workgroup key split: steps of up to kSplitRows rows, up to kMaxSplits splits per (row, head)
size_t stack_attn_workspace_floats(int32_t heads, int32_t maps, int32_t vdim)
{
    return (size_t) kSplitRows * heads * kMaxSplits * maps * (vdim + 2);
}

// the tile kernel's shapes: bfloat16, dim 32 / 64 / 128, vdim 32 / 64 / 128 (one map: dim 96 / 192 and vdim 96 as well), pages of a multiple
// of 32 keys
bool stack_attention_tiled(const StackAttnParams& p)
{
    const bool one = p.maps == 1;
    const bool std_shape = (p.dim == 32 || p.dim == 64 || p.dim == 128 || (one && (p.dim == 96 || p.dim == 192)))
        && (p.vdim == 32 || p.vdim == 64 || p.vdim == 128 || (one && p.vdim == 96));
    const bool latent_shape = p.maps == 1 && p.kv_heads == 1 && ((p.dim == 160 && p.vdim == 128) || (p.dim == 320 && p.vdim == 256)
                                  || (p.dim == p.vdim && (p.dim == 96 || p.dim == 192 || p.dim == 256)));
    // what only the general kernels do: head-mixed weights, a gate per channel, kept first keys under a window
    if (p.talk || (p.out_gate && p.gate_wide))
        return false;
    return p.dtype == DT_BF16 && (std_shape || latent_shape) && p.page % 32 == 0 && p.max_count > 0 && p.entries > 0 && !(reinterpret_cast<uintptr_t>(p.q) & 15)
        && !(reinterpret_cast<uintptr_t>(p.k_pool) & 15) && !(reinterpret_cast<uintptr_t>(p.v_pool) & 7);
}

int launch_stack_attention(const StackAttnParams& p, hipStream_t stream)
{
    if (p.tokens <= 0)
        return 0;
    static const bool general_only = [] {
        const char* v = std::getenv("TLLM_STACK_ATTN_GENERAL"); // measurement knob: 1 = every shape on the general kernel
        return v && v[0] == '1';
    }();
    if (!general_only && p.talk && p.pair_ws && p.maps == 1 && p.heads >= 1 && p.kv_heads >= 1 && p.heads % p.kv_heads == 0)
    {
        // head-mixed weights on the tile kernels: every query head's weights over every value head's rows (kv_heads x the pairs of a
        // plain launch), then the mixing as a sum over those terms - the mixing is linear in the weights, so it commutes with P V
        StackAttnParams c = p;
        c.talk = nullptr;
        c.out_gate = nullptr;
        c.heads = p.heads * p.kv_heads;
        c.cross_values = 1;
        c.out = p.pair_ws;
        if (stack_attention_tiled(c))
        {
            const int rc = launch_tile_d<1>(c, stream);
            if (rc < 0)
                return rc;
            if (rc == 0)
                return launch_stack_talk_combine(p, p.pair_ws, stream);
        }
    }
    if (!general_only && p.heads >= 1 && p.kv_heads >= 1 && p.heads % p.kv_heads == 0 && stack_attention_tiled(p))
    {
        int rc = p.maps == 2 ? launch_tile_d<2>(p, stream) : (p.maps == 1 ? launch_tile_d<1>(p, stream) : 1);
        if (rc == 1 && p.maps == 1)
            rc = launch_tile_latent(p, stream);
        if (rc <= 0)
            return rc;
    }
    return launch_stack_attention_general(p, stream);
}

} // namespace kernels
} // namespace tllm
