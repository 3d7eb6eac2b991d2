// The recurrences of the stack engine's state layers (HGRN2, gated delta rule, Mamba-2) over prompts, 16 rows at a time.
//
// All three are  S <- diag(f_t) S + k_t u_t^T,  o_t = S^T q_t  with a state S [D, V] per head in fp32 (HGRN2: u = v, k = 1 - f; delta rule: u_t =
// beta_t (v_t - (diag(f_t) S)^T k_t); Mamba-2: one f per head, k = dt B, u = x).  Row by row that is a chain of rows: 1.0 ms for 1024 rows
// whatever the width, the chip idle (a row took 1 us of dependent latency).  With b_t = f_1 ... f_t inside a chunk of 16 rows,
//   o_t = (b_t q_t)^T S_0 + sum_{s <= t} P[t, s] u_s,   P[t, s] = sum_d q_t[d] k_s[d] f_{s+1}[d] ... f_t[d]
//   S_16 = b_16 S_0 + sum_s (k_s f_{s+1} ... f_16) u_s^T
//   delta rule:  u = T (v - (b k)^T S_0),  T = (I + diag(beta) M)^-1 diag(beta),  M[t, s] = sum_d k_t[d] k_s[d] f_{s+1}[d] ... f_t[d], s < t
// so only S_0 -> S_16 is a chain, of matrix products.  Every decay is a product of the factors between two rows (never a quotient of cumulative
// products: nothing underflows into 0 / 0 whatever the gates), all sums are fp32 (v_mfma_f32_16x16x4_f32, no reduced-precision matrix
// mode) in both element types.
//
// Two launches.  chunk_prepare_kernel / ssm_prepare_kernel: a workgroup per (chunk, head), resp. (chunk, group), all chunks at once: gates, unit
// norms, the decayed vectors, P, M and T into scratch.  Then a workgroup per (entry, head, 16 columns of V) walks the chunks; its waves keep the
// state's rows, 16 at a time, in registers in the MFMA's accumulator layout (lane: column lane & 15, rows 4 (lane >> 4) + i), which is also its
// B-operand layout when the four K = 4 steps of 16 rows take rows 4 g + i in step i: S, u and v go from product to product without moving, and what
// comes from scratch is 16 bytes per lane.  chunk_walk_kernel (HGRN2 and Mamba-2) and delta_chunk_walk_kernel: four waves, which take the state's 16
// rows in turn, and one barrier per chunk, where their partial o (and S^T k) meet; the next chunk's operands are in flight under this one's products.
// eight_chunk_walk_kernel (HGRN2 and Mamba-2, long portions in few workgroups: eight_chunks_serve): eight waves, one to 16 rows, and a barrier per
// eight chunks.
//
// Measured (us, both launches, 16 heads): HGRN2 128 x 128, 1024 rows 1024 -> 57; delta rule 128 x 128, three prompts of 683 rows in all 1740 1193 -> 109;
// Mamba-2 64 heads 128 x 64, 1021 rows 400 -> 57.
#include "dev_utils.h"
#include "launch_util.h"
#include "stack_chunk.h"
#include "stack_kernels.h"
#include <algorithm>
#include <type_traits>

namespace tllm
{
namespace kernels
{
using namespace dev;

namespace
{
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int DT>
__device__ __forceinline__ float ld_el(const void* p, int64_t i)
{
    if constexpr (DT == DT_BF16)
        return bf2f(reinterpret_cast<const uint16_t*>(p)[i]);
    else
        return reinterpret_cast<const float*>(p)[i];
}

constexpr int HGRN = CHUNK_HGRN2, DELTA = CHUNK_DELTA, SSM = CHUNK_SSM;

// What the three kinds have in common, filled by the launchers below.
struct ChunkArgs
{
    int32_t heads = 0, D = 0, V = 0, groups = 1, entries = 0, slots = 0;
    int32_t max_count = 0; // rows of the longest entry
    // HGRN: q at proj column h D, f at heads D + h D, v at 2 heads D + h V.  DELTA: x = [q | k | v].  SSM: xbc = [x | B | C], proj = [z | ... | dt]
    const void* proj = nullptr;
    int64_t ldp = 0;
    const void* xbc = nullptr;
    int64_t ldx = 0;
    int32_t qk_heads = 0;
    const float* f_bias = nullptr; // HGRN
    const float* lower = nullptr;
    const float* decay_raw = nullptr; // DELTA
    const float* dt_bias = nullptr;   // DELTA, SSM
    const float* a_log = nullptr;
    const void* beta_raw = nullptr;
    int64_t ld_beta = 0;
    const float* d_skip = nullptr; // SSM
    float* state = nullptr;
    float* out = nullptr; // [tokens, heads V]
    const int32_t* ent_slot = nullptr;
    const int32_t* ent_first = nullptr;
    const int32_t* ent_count = nullptr;
    const int32_t* ent_pos0 = nullptr;
    // scratch, by chunk slot c and head: the slot of an entry's chunk j is ent_first / 16 + entry + j
    float* qt = nullptr; // [c][heads | groups][16][D]  b_t q_t, SSM: C
    float* kb = nullptr; // [c][heads][16][D]  b_t k_t                        (DELTA)
    float* kt = nullptr; // [c][heads | groups][D][16]  k_s f_{s+1} ... f_16, SSM: B transposed
    float* pm = nullptr; // [c][heads][16][16] P
    float* tm = nullptr; // [c][heads][16][16] T                              (DELTA)
    float* bc = nullptr; // [c][heads][D] f_1 ... f_16; SSM: [c][heads][48] = {b_t}, {dt_s f_{s+1} ... f_16}, f_1 ... f_16 in [32]
};

// entry and chunk of a slot; false where the slot belongs to none
__device__ __forceinline__ bool find_chunk(const ChunkArgs& a, int slot, int& e, int& j)
{
    const int lane = threadIdx.x & 63;
    for (int e0 = 0; e0 < a.entries; e0 += 64)
    {
        const int i = e0 + lane;
        int at = 0, n = 0;
        if (i < a.entries)
        {
            at = a.ent_first[i] / CHUNK_ROWS + i;
            n = (a.ent_count[i] + CHUNK_ROWS - 1) / CHUNK_ROWS;
        }
        const uint64_t mine = __ballot(slot >= at && slot < at + n);
        if (mine)
        {
            const int l = __ffsll((unsigned long long) mine) - 1;
            e = e0 + l;
            j = slot - __shfl(at, l, 64);
            return true;
        }
    }
    return false;
}

__device__ __forceinline__ float sigmoid_f(float z)
{
    return 1.f / (1.f + expf(-z));
}
__device__ __forceinline__ float softplus_f(float z)
{
    return z > 20.f ? z : log1pf(expf(z));
}
// exp(-rate softplus(z)) as the row-by-row kernel takes it (stack_delta.hip)
template <int DT>
__device__ __forceinline__ float decay_of(float rate, float z)
{
    if constexpr (DT == DT_BF16)
    {
        constexpr float LOG2E = 1.4426950408889634f;
        const float sp2 = z > 20.f ? z * LOG2E : __builtin_amdgcn_logf(1.f + __builtin_amdgcn_exp2f(z * LOG2E));
        return __builtin_amdgcn_exp2f(-rate * sp2);
    }
    else
        return expf(-rate * softplus_f(z));
}

constexpr int R = CHUNK_ROWS;

// HGRN2 and delta rule: a workgroup per (chunk, head), D a multiple of 64 up to 256
// (Rows 0 .. 7 of a chunk meet eight rows of it in the delta rule's P and M, not sixteen, which needs 72 registers if the compiler is held to them: left to itself it takes 82, five
// workgroups on a CU for six.  us, 16 heads of 128 x 128, 1021 rows, 16 rows always / 82 registers / 72: 25.7 / 24.6 / 24.6; 24 heads, four times 1021 101 / 109 / 98.  HGRN2's P alone is
// quicker the long way: 32 heads, four times 1021 97 and 105.)
template <int DT, int MODE>
__global__ __launch_bounds__(256, MODE == DELTA ? 6 : 1) void chunk_prepare_kernel(const ChunkArgs a)
{
    extern __shared__ __attribute__((aligned(16))) float sm[];
    const int D = a.D, h = blockIdx.y, slot = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    int e, j;
    if (!find_chunk(a, slot, e, j))
        return;
    const int t0 = a.ent_first[e] + j * R, nt = min(R, a.ent_count[e] - j * R);
    float* fs = sm;          // [R][D] decay
    float* ks = fs + R * D;  // [R][D]
    float* qs = ks + R * D;  // [R][D]
    float* ms = qs + R * D;  // [R][R] M
    float* bs = ms + R * R;  // [R] beta
    const int hk = MODE == DELTA ? h / (a.heads / a.qk_heads) : 0;
    const float rate = MODE == DELTA ? expf(a.a_log[h]) : 0.f;
    for (int i = tid; i < R * D; i += 256)
    {
        const int t = i / D, d = i % D;
        float f = 1.f, k = 0.f, q = 0.f; // a row past the entry's end leaves the state as it is
        if (t < nt)
        {
            const int64_t r = t0 + t;
            if constexpr (MODE == HGRN)
            {
                q = ld_el<DT>(a.proj, r * a.ldp + h * D + d);
                q = q / (1.f + expf(-q));
                if (DT == DT_BF16)
                    q = bf2f(f2bf(q)); // the projection's activation is a bfloat16 value; everything behind it is fp32
                const float lo = a.lower[h * D + d];
                f = lo + (1.f - lo) * sigmoid_f(ld_el<DT>(a.proj, r * a.ldp + (a.heads + h) * D + d) + a.f_bias[h * D + d]);
                k = 1.f - f;
            }
            else
            {
                q = ld_el<DT>(a.xbc, r * a.ldx + hk * D + d);
                k = ld_el<DT>(a.xbc, r * a.ldx + (a.qk_heads + hk) * D + d);
                f = decay_of<DT>(rate, a.decay_raw[r * a.heads * D + h * D + d] + a.dt_bias[h * D + d]);
            }
        }
        fs[i] = f;
        ks[i] = k;
        qs[i] = q;
    }
    if (MODE == DELTA && tid < R)
        bs[tid] = tid < nt ? sigmoid_f(ld_el<DT>(a.beta_raw, (int64_t) (t0 + tid) * a.ld_beta + h)) : 0.f;
    __syncthreads();
    if constexpr (MODE == DELTA)
    {
        // unit q (times dim^-1/2) and k: a wave per row
        for (int t = wid; t < R; t += 4)
        {
            float sq = 0.f, sk = 0.f;
            for (int d = lane; d < D; d += 64)
            {
                sq = fmaf(qs[t * D + d], qs[t * D + d], sq);
                sk = fmaf(ks[t * D + d], ks[t * D + d], sk);
            }
            const float iq = 1.f / (sqrtf((float) D) * sqrtf(wave_sum(sq) + 1e-6f)), ik = 1.f / sqrtf(wave_sum(sk) + 1e-6f);
            for (int d = lane; d < D; d += 64)
            {
                qs[t * D + d] *= iq;
                ks[t * D + d] *= ik;
            }
        }
        __syncthreads();
    }
    const int64_t ch = (int64_t) slot * a.heads + h;
    // P and M: thread (row pair, channel pair): rows tp and 15 - tp against every row s, the decay between them built up as s goes down
    {
        const int dg = tid & 31, tp = tid >> 5;
#pragma unroll
        for (int half = 0; half < 2; ++half)
        {
            const int t = half ? R - 1 - tp : tp, rows = MODE != DELTA || half ? R : R / 2; // (unrolled, as is half)
            float pa[R], ma[R];
#pragma unroll
            for (int s = 0; s < R; ++s)
                pa[s] = ma[s] = 0.f;
            for (int d = dg * 2; d < D; d += 64)
            {
                float2 q = *reinterpret_cast<const float2*>(qs + t * D + d), k = *reinterpret_cast<const float2*>(ks + t * D + d);
#pragma unroll
                for (int s = rows - 1; s >= 0; --s)
                {
                    if (s > t)
                        continue;
                    const float2 ksv = *reinterpret_cast<const float2*>(ks + s * D + d), f = *reinterpret_cast<const float2*>(fs + s * D + d);
                    pa[s] = fmaf(q.x, ksv.x, fmaf(q.y, ksv.y, pa[s]));
                    if (MODE == DELTA)
                    {
                        ma[s] = fmaf(k.x, ksv.x, fmaf(k.y, ksv.y, ma[s]));
                        k.x *= f.x;
                        k.y *= f.y;
                    }
                    q.x *= f.x; // q_t f_s ... f_t meets k_{s - 1}
                    q.y *= f.y;
                }
            }
#pragma unroll
            for (int s = 0; s < rows; ++s)
            {
                pa[s] = group_sum<32>(pa[s]);
                if (MODE == DELTA)
                    ma[s] = group_sum<32>(ma[s]);
            }
            if (dg == 0)
            {
#pragma unroll
                for (int s = 0; s < R; s += 4)
                {
                    *reinterpret_cast<float4*>(a.pm + ch * R * R + t * R + s) = make_float4(pa[s], pa[s + 1], pa[s + 2], pa[s + 3]);
                    if (MODE == DELTA)
                        *reinterpret_cast<float4*>(ms + t * R + s) = make_float4(ma[s], ma[s + 1], ma[s + 2], ma[s + 3]);
                }
            }
        }
    }
    // the decayed vectors: forward from the chunk's start, backward from its end
    for (int i = tid; i < 2 * D; i += 256)
    {
        const int d = i % D;
        float w = 1.f;
        if (i < D)
        {
#pragma unroll
            for (int t = 0; t < R; ++t)
            {
                w *= fs[t * D + d];
                a.qt[(ch * R + t) * D + d] = qs[t * D + d] * w;
                if (MODE == DELTA)
                    a.kb[(ch * R + t) * D + d] = ks[t * D + d] * w;
            }
            a.bc[ch * D + d] = w;
        }
        else
        {
            float o[R];
#pragma unroll
            for (int s = R - 1; s >= 0; --s)
            {
                o[s] = ks[s * D + d] * w;
                w *= fs[s * D + d];
            }
#pragma unroll
            for (int s = 0; s < R; s += 4)
                *reinterpret_cast<float4*>(a.kt + (ch * D + d) * R + s) = make_float4(o[s], o[s + 1], o[s + 2], o[s + 3]);
        }
    }
    if constexpr (MODE == DELTA)
    {
        __syncthreads();
        // T by forward substitution, a thread per column
        if (tid < R)
        {
            float x[R];
#pragma unroll
            for (int i = 0; i < R; ++i)
            {
                float s0 = 0.f;
#pragma unroll
                for (int s = 0; s < i; ++s)
                    s0 = fmaf(ms[i * R + s], x[s], s0);
                x[i] = (i == tid ? 1.f : 0.f) - bs[i] * s0;
            }
#pragma unroll
            for (int i = 0; i < R; ++i)
                a.tm[ch * R * R + i * R + tid] = x[i] * bs[tid];
        }
    }
}

// Mamba-2: a workgroup per (chunk, group): B transposed, C B^T once for the group's heads, then each head's decays
template <int DT>
__global__ __launch_bounds__(256) void ssm_prepare_kernel(const ChunkArgs a)
{
    extern __shared__ __attribute__((aligned(16))) float sm[];
    const int D = a.D, g = blockIdx.y, slot = blockIdx.x, tid = threadIdx.x;
    int e, j;
    if (!find_chunk(a, slot, e, j))
        return;
    const int t0 = a.ent_first[e] + j * R, nt = min(R, a.ent_count[e] - j * R);
    const int per = a.heads / a.groups, inner = a.heads * a.V, GN = a.groups * D, DP = D + 4;
    float* bs = sm;            // [R][DP] (a row's end is padded: the rows of a column then fall on different banks)
    float* cs = bs + R * DP;   // [R][DP]
    float* dts = cs + R * DP;  // [per][R] step size
    float* fs = dts + per * R; // [per][R] decay
    for (int i = tid; i < R * D; i += 256)
    {
        const int t = i / D, d = i % D;
        const int64_t r = t0 + min(t, nt - 1);
        const float c = ld_el<DT>(a.xbc, r * a.ldx + inner + GN + g * D + d);
        bs[t * DP + d] = ld_el<DT>(a.xbc, r * a.ldx + inner + g * D + d);
        cs[t * DP + d] = c;
        a.qt[((int64_t) slot * a.groups + g) * R * D + i] = c;
    }
    for (int i = tid; i < per * R; i += 256)
    {
        const int h = g * per + i / R, t = i % R;
        float dt = 0.f, f = 1.f; // a row past the entry's end leaves the state as it is
        if (t < nt)
        {
            dt = softplus_f(ld_el<DT>(a.proj, (int64_t) (t0 + t) * a.ldp + 2 * inner + 2 * GN + h) + a.dt_bias[h]);
            f = expf(-expf(a.a_log[h]) * dt);
        }
        dts[i] = dt;
        fs[i] = f;
    }
    __syncthreads();
    const int64_t cg = (int64_t) slot * a.groups + g;
    for (int i = tid; i < D * (R / 4); i += 256)
    {
        const int d = i / (R / 4), s = i % (R / 4) * 4;
        *reinterpret_cast<float4*>(a.kt + (cg * D + d) * R + s) = make_float4(bs[s * DP + d], bs[(s + 1) * DP + d], bs[(s + 2) * DP + d], bs[(s + 3) * DP + d]);
    }
    const int t = tid >> 4, s = tid & 15;
    float cb[4] = {0.f, 0.f, 0.f, 0.f};
    for (int d = 0; d < D; d += 4)
    {
        const float4 c4 = *reinterpret_cast<const float4*>(cs + t * DP + d), b4 = *reinterpret_cast<const float4*>(bs + s * DP + d);
        cb[0] = fmaf(c4.x, b4.x, cb[0]);
        cb[1] = fmaf(c4.y, b4.y, cb[1]);
        cb[2] = fmaf(c4.z, b4.z, cb[2]);
        cb[3] = fmaf(c4.w, b4.w, cb[3]);
    }
    const float dot = (cb[0] + cb[1]) + (cb[2] + cb[3]);
    for (int i = 0; i < per; ++i)
    {
        const int64_t ch = (int64_t) slot * a.heads + g * per + i;
        float w = s <= t ? dts[i * R + s] : 0.f;
        for (int k = s + 1; k <= t; ++k)
            w *= fs[i * R + k];
        a.pm[ch * R * R + tid] = s <= t ? dot * w : 0.f; // (the dot of an overflowed row times 0 is no 0)
    }
    for (int i = tid; i < per * R; i += 256)
    {
        const int hh = i / R, tt = i % R;
        float b = 1.f, w = dts[i];
        for (int k = 0; k <= tt; ++k)
            b *= fs[hh * R + k];
        for (int k = tt + 1; k < R; ++k)
            w *= fs[hh * R + k];
        float* o = a.bc + ((int64_t) slot * a.heads + g * per + hh) * 48;
        o[tt] = b;
        o[R + tt] = w;
        if (tt == R - 1)
            o[2 * R] = b;
    }
}

// whether any lane of the wave holds an infinity, a NaN or a value near them
__device__ __forceinline__ bool any_large(const f32x4& x)
{
    return __builtin_amdgcn_ballot_w64(!((fabsf(x[0]) + fabsf(x[1])) + (fabsf(x[2]) + fabsf(x[3])) < 1e30f)) != 0;
}
__device__ __forceinline__ float pick(const f32x4& x, int i)
{
    return i < 2 ? (i ? x[1] : x[0]) : (i == 2 ? x[2] : x[3]);
}

// acc + M x of a lower triangular M [16, 16] (A-operand layout: M[lane & 15][4 (lane >> 4) + j] in element j) and x (B-operand layout: row
// 4 (lane >> 4) + j), j in [j0, j1), over the rows s <= t alone
__device__ __forceinline__ f32x4 lower_product(const f32x4& m, const f32x4& x, int j0, int j1, f32x4 acc)
{
    const int lane = threadIdx.x & 63, g4 = lane >> 4;
#pragma unroll 1
    for (int g = 0; g < 4; ++g)
#pragma unroll 1
        for (int j = j0; j < j1; ++j)
        {
            const float mj = pick(m, j), xs = __shfl(pick(x, j), (lane & 15) + 16 * g, 64);
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                const int t = 4 * g4 + i;
                const float mt = __shfl(mj, t + 16 * g, 64);
                acc[i] = 4 * g + j <= t ? fmaf(mt, xs, acc[i]) : acc[i];
            }
        }
    return acc;
}

// HGRN2 and Mamba-2 where eight_chunks_serve says no.  One workgroup per (entry, head, 16 columns of V): TILES * 64 rows of state (D), wave w keeps rows 16 (w + 4 j) .. + 16
template <int DT, int MODE, int TILES>
__global__ __launch_bounds__(256) void chunk_walk_kernel(const ChunkArgs a)
{
    static_assert(MODE != DELTA, "delta_chunk_walk_kernel");
    __shared__ f32x4 po[2][4][64];
    constexpr int D = TILES * 64;
    const int e = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int c16 = lane & 15, g4 = lane >> 4;
    const int v = blockIdx.z * 16 + c16, V = a.V, vc = v < V ? v : V - 1;
    const int first = a.ent_first[e], count = a.ent_count[e], nchunk = (count + R - 1) / R;
    const int64_t slot0 = first / R + e;
    const int grp = MODE == SSM ? h / (a.heads / a.groups) : 0;
    float* st = a.state + ((int64_t) a.ent_slot[e] * a.heads + h) * D * V;
    const bool live = v < V, carry = a.ent_pos0[e] > 0;

    f32x4 S[TILES];
#pragma unroll
    for (int j = 0; j < TILES; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            S[j][i] = live && carry ? st[(int64_t) (16 * (wid + 4 * j) + 4 * g4 + i) * V + v] : 0.f;
    const float dsk = MODE == SSM ? a.d_skip[h] : 0.f;

    // a chunk's operands as this lane holds them; `raw` ones are converted where they are used, so that nothing waits at its load
    typedef typename std::conditional<DT == DT_BF16, uint16_t, float>::type Raw;
    struct Ops
    {
        f32x4 q[TILES], kt[TILES], b[MODE == SSM ? 1 : TILES], p;
        f32x4 bt, ws; // SSM: b_t of this lane's rows, dt_s f_{s+1} ... f_16
        Raw v[4], z;
        float b16;
    };
    const Raw* vsrc = reinterpret_cast<const Raw*>(MODE == HGRN ? a.proj : a.xbc);
    const int64_t vld = MODE == HGRN ? a.ldp : a.ldx;
    const int64_t vcol = (MODE == HGRN ? 2 * a.heads * D : 0) + h * V + vc;
    auto request = [&](int j, Ops& o) {
        const int64_t slot = slot0 + j, ch = slot * a.heads + h, kg = MODE == SSM ? slot * a.groups + grp : ch;
#pragma unroll
        for (int n = 0; n < TILES; ++n)
        {
            const int d0 = 16 * (wid + 4 * n);
            o.kt[n] = *reinterpret_cast<const f32x4*>(a.kt + (kg * D + d0 + c16) * R + 4 * g4);
            o.q[n] = *reinterpret_cast<const f32x4*>(a.qt + (kg * R + c16) * D + d0 + 4 * g4);
            if constexpr (MODE != SSM)
                o.b[n] = *reinterpret_cast<const f32x4*>(a.bc + ch * D + d0 + 4 * g4);
        }
        o.p = *reinterpret_cast<const f32x4*>(a.pm + ch * R * R + c16 * R + 4 * g4);
        if constexpr (MODE == SSM)
        {
            o.bt = *reinterpret_cast<const f32x4*>(a.bc + ch * 48 + 4 * g4);
            o.ws = *reinterpret_cast<const f32x4*>(a.bc + ch * 48 + R + 4 * g4);
            o.b16 = a.bc[ch * 48 + 2 * R];
            o.z = reinterpret_cast<const Raw*>(a.proj)[(int64_t) (first + min(j * R + 4 * g4 + wid, count - 1)) * a.ldp + h * V + vc];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            o.v[i] = vsrc[(int64_t) (first + min(j * R + 4 * g4 + i, count - 1)) * vld + vcol];
    };
    auto cvt = [](Raw r) -> float {
        if constexpr (DT == DT_BF16)
            return bf2f(r);
        else
            return r;
    };

    auto chunk = [&](int j, const Ops& o) {
        const int buf = j & 1;
        f32x4 u;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            u[i] = cvt(o.v[i]);
        // two sums per product: a product's next step waits for the one before
        f32x4 acc = {0.f, 0.f, 0.f, 0.f}, acc1 = acc;
#pragma unroll
        for (int n = 0; n < TILES; ++n)
#pragma unroll
            for (int i = 0; i < 4; i += 2)
            {
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(o.q[n][i], S[n][i], acc, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(o.q[n][i + 1], S[n][i + 1], acc1, 0, 0, 0);
            }
        acc = acc + acc1;
        if constexpr (MODE == SSM)
            acc = acc * o.bt;
        const f32x4 past = acc; // what the rows ahead of the chunk give
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(pick(o.p, wid), pick(u, wid), acc, 0, 0, 0); // this wave's quarter of P u
        po[buf][wid][lane] = acc;
        __syncthreads();
#pragma unroll
        for (int n = 0; n < TILES; ++n)
        {
            if constexpr (MODE == SSM)
                S[n] = S[n] * o.b16;
            else
                S[n] = S[n] * o.b[n];
        }
        const f32x4 us = MODE == SSM ? u * o.ws : u;
#pragma unroll
        for (int n = 0; n < TILES; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                S[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.kt[n][i], us[i], S[n], 0, 0, 0);
        // wave w finishes rows 4 g + w
        const float* pf = reinterpret_cast<const float*>(&po[buf][0][0]);
        auto waves_sum = [&] { return (pf[lane * 4 + wid] + pf[256 + lane * 4 + wid]) + (pf[512 + lane * 4 + wid] + pf[768 + lane * 4 + wid]); };
        float y = waves_sum();
        // The zeros of P above its diagonal meet every row in a matrix product, and 0 times an infinity or a NaN is a NaN: where a row
        // has one, the outputs are formed again row by row, without what follows a row (the state takes every row in any case).  All waves hold
        // the same u, so that the branch is the workgroup's.
        // Asked behind the chunk's products: a branch among them takes the next request's addresses and the state's factors out of their
        // shadow, 60 us for the walk of HGRN2 128 x 128 over 1024 rows instead of 50.
        if (any_large(u))
        {
            __syncthreads(); // (every wave has read the sums above)
            po[buf][wid][lane] = lower_product(o.p, u, wid, wid + 1, past);
            __syncthreads();
            y = waves_sum();
        }
        const int row = j * R + 4 * g4 + wid;
        if constexpr (MODE == SSM)
        {
            const float z = cvt(o.z);
            y = fmaf(dsk, pick(u, wid), y) * (z / (1.f + expf(-z)));
        }
        if (live && row < count)
            a.out[(int64_t) (first + row) * (a.heads * V) + h * V + v] = y;
    };

    // Three sets of operands: a chunk's are requested two chunks ahead.  Every request is made (past the end the last chunk's once more): one
    // under a condition would have the compiler wait as if it had not been made, for all that is in flight.
    const int last = nchunk - 1;
    if (last < 0)
        return;
    Ops o0, o1, o2;
    request(0, o0);
    request(min(1, last), o1);
    for (int j = 0;; j += 3)
    {
        request(min(j + 2, last), o2);
        chunk(j, o0);
        if (j + 1 > last)
            break;
        request(min(j + 3, last), o0);
        chunk(j + 1, o1);
        if (j + 2 > last)
            break;
        request(min(j + 4, last), o1);
        chunk(j + 2, o2);
        if (j + 3 > last)
            break;
    }
    if (live)
    {
#pragma unroll
        for (int j = 0; j < TILES; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                st[(int64_t) (16 * (wid + 4 * j) + 4 * g4 + i) * V + v] = S[j][i];
    }
}

// The walk of the delta rule, whose u hangs on the state: one workgroup per (entry, head, 16 columns of V), wave w keeps rows 16 (w + 4 j) .. + 16 of the state.  The chain of a chunk is
// (b k)^T S of a wave's rows, their sum over the waves through LDS, T on what is left of v, and S's update; everything else stands beside it: q's product with S covers the way
// through LDS, a wave adds its quarter of P u to it, and the sums over the waves become outputs a chunk later, behind that chunk's one barrier.  With everything in the order of the formulas
// and three sets of operands 1.35 us a chunk where a CU has one workgroup, here 1.15 (a chunk brings 27 KB).  Both launches, us, in brackets that form: 16 heads 128 x 128, one prompt of 683 rows 67 (76), three of
// 1672 in all 96 (108), 24 heads 136 (158), eight of 240 92 (100).  32 columns a workgroup, which halve what its operands bring, made the chain longer: 109, 120, 167, 89.
template <int DT, int TILES>
__global__ __launch_bounds__(256, 2) void delta_chunk_walk_kernel(const ChunkArgs a)
{
    __shared__ f32x4 po[2][4][64], pr[2][4][64];
    constexpr int D = TILES * 64;
    const int e = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c16 = lane & 15, g4 = lane >> 4;
    const int v = blockIdx.z * 16 + c16, V = a.V, vc = v < V ? v : V - 1;
    const int first = a.ent_first[e], count = a.ent_count[e], last = (count + R - 1) / R - 1;
    if (last < 0)
        return;
    const int64_t slot0 = first / R + e;
    float* st = a.state + ((int64_t) a.ent_slot[e] * a.heads + h) * D * V;
    const bool live = v < V, carry = a.ent_pos0[e] > 0;

    f32x4 S[TILES];
#pragma unroll
    for (int j = 0; j < TILES; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            S[j][i] = live && carry ? st[(int64_t) (16 * (wid + 4 * j) + 4 * g4 + i) * V + v] : 0.f;

    // a chunk's operands as this lane holds them; `raw` ones are converted where they are used, so that nothing waits at its load
    typedef typename std::conditional<DT == DT_BF16, uint16_t, float>::type Raw;
    struct Ops
    {
        f32x4 q[TILES], kb[TILES], kt[TILES], b[TILES], p, t;
        Raw v[4];
    };
    const Raw* vsrc = reinterpret_cast<const Raw*>(a.xbc) + 2 * a.qk_heads * D + h * V + vc;
    const int64_t vrow0 = (int64_t) first * a.ldx;
    auto request_kb = [&](int j, Ops& o) {
        const float* kb = a.kb + ((slot0 + j) * a.heads + h) * R * D;
#pragma unroll
        for (int n = 0; n < TILES; ++n)
            o.kb[n] = *reinterpret_cast<const f32x4*>(kb + c16 * D + 16 * (wid + 4 * n) + 4 * g4);
    };
    auto request_q = [&](int j, Ops& o) {
        const float* q = a.qt + ((slot0 + j) * a.heads + h) * R * D;
#pragma unroll
        for (int n = 0; n < TILES; ++n)
            o.q[n] = *reinterpret_cast<const f32x4*>(q + c16 * D + 16 * (wid + 4 * n) + 4 * g4);
    };
    auto request_v = [&](int j, Ops& o) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            o.v[i] = vsrc[vrow0 + (int64_t) min(j * R + 4 * g4 + i, count - 1) * a.ldx];
        o.t = *reinterpret_cast<const f32x4*>(a.tm + ((slot0 + j) * a.heads + h) * R * R + c16 * R + 4 * g4);
    };
    auto request_k = [&](int j, Ops& o) {
        const int64_t ch = (slot0 + j) * a.heads + h;
#pragma unroll
        for (int n = 0; n < TILES; ++n)
        {
            o.b[n] = *reinterpret_cast<const f32x4*>(a.bc + ch * D + 16 * (wid + 4 * n) + 4 * g4);
            o.kt[n] = *reinterpret_cast<const f32x4*>(a.kt + (ch * D + 16 * (wid + 4 * n) + c16) * R + 4 * g4);
        }
        o.p = *reinterpret_cast<const f32x4*>(a.pm + ch * R * R + c16 * R + 4 * g4);
    };
    auto cvt = [](Raw r) -> float {
        if constexpr (DT == DT_BF16)
            return bf2f(r);
        else
            return r;
    };
    // wave w finishes rows 4 g + w of chunk j, behind a barrier that its sums are ahead of
    auto finish = [&](int j) {
        const float* pf = reinterpret_cast<const float*>(&po[j & 1][0][0]);
        const float y = (pf[lane * 4 + wid] + pf[256 + lane * 4 + wid]) + (pf[512 + lane * 4 + wid] + pf[768 + lane * 4 + wid]);
        const int row = j * R + 4 * g4 + wid;
        if (live && row < count)
            a.out[(int64_t) (first + row) * (a.heads * V) + h * V + v] = y;
    };

    auto chunk = [&](int j, int buf, Ops& o) {
        const int next = min(j + 2, last);
        // two sums per product: a product's next step waits for the one before
        f32x4 accr = {0.f, 0.f, 0.f, 0.f}, accr1 = accr, acc = accr, acc1 = accr;
#pragma unroll
        for (int n = 0; n < TILES; ++n)
#pragma unroll
            for (int i = 0; i < 4; i += 2)
            {
                accr = __builtin_amdgcn_mfma_f32_16x16x4f32(o.kb[n][i], S[n][i], accr, 0, 0, 0);
                accr1 = __builtin_amdgcn_mfma_f32_16x16x4f32(o.kb[n][i + 1], S[n][i + 1], accr1, 0, 0, 0);
            }
        pr[buf][wid][lane] = accr + accr1;
        __builtin_amdgcn_sched_barrier(0);
        request_kb(next, o);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        const f32x4 r0 = pr[buf][0][lane], r1 = pr[buf][1][lane], r2 = pr[buf][2][lane], r3 = pr[buf][3][lane];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = 0; n < TILES; ++n)
#pragma unroll
            for (int i = 0; i < 4; i += 2)
            {
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(o.q[n][i], S[n][i], acc, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(o.q[n][i + 1], S[n][i + 1], acc1, 0, 0, 0);
            }
        __builtin_amdgcn_sched_barrier(0);
        f32x4 x;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            x[i] = cvt(o.v[i]) - ((r0[i] + r1[i]) + (r2[i] + r3[i]));
        f32x4 u = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i)
            u = __builtin_amdgcn_mfma_f32_16x16x4f32(o.t[i], x[i], u, 0, 0, 0);
        acc = acc + acc1;
#pragma unroll
        for (int n = 0; n < TILES; ++n)
            S[n] = S[n] * o.b[n];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int n = 0; n < TILES; ++n)
                S[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.kt[n][i], u[i], S[n], 0, 0, 0);
        f32x4 part = __builtin_amdgcn_mfma_f32_16x16x4f32(pick(o.p, wid), pick(u, wid), acc, 0, 0, 0); // with this wave's quarter of P u
        // The zeros of P and T above their diagonals meet every row in a matrix product, and 0 times an infinity or a NaN is a NaN: where a row
        // has one, P u is formed again row by row, without what follows a row (the state takes every row in any case).  All waves hold
        // the same x.  (u overflows only where x is near it, T's entries are below 2^15.)
        if (any_large(x))
        {
            const f32x4 none = {0.f, 0.f, 0.f, 0.f};
            part = wid == 0 ? lower_product(o.p, lower_product(o.t, x, 0, 4, none), 0, 4, acc) : acc;
        }
        po[buf][wid][lane] = part;
        __builtin_amdgcn_sched_barrier(0);
        request_q(next, o);
        __builtin_amdgcn_sched_barrier(0);
        request_v(next, o);
        __builtin_amdgcn_sched_barrier(0);
        request_k(next, o);
        __builtin_amdgcn_sched_barrier(0);
        if (j > 0)
            finish(j - 1);
    };

    // Two sets of operands, each requested again as it is used, two chunks ahead and in that order: the waits count.  Every request is made (past the end the last chunk's once more):
    // one under a condition would have the compiler wait as if it had not been made, for all that is in flight.
    Ops o0, o1;
    auto request = [&](int j, Ops& o) {
        request_kb(j, o);
        __builtin_amdgcn_sched_barrier(0);
        request_q(j, o);
        __builtin_amdgcn_sched_barrier(0);
        request_v(j, o);
        __builtin_amdgcn_sched_barrier(0);
        request_k(j, o);
        __builtin_amdgcn_sched_barrier(0);
    };
    request(0, o0);
    request(min(1, last), o1);
    for (int j = 0;; j += 2)
    {
        chunk(j, 0, o0);
        if (j + 1 > last)
            break;
        chunk(j + 1, 1, o1);
        if (j + 2 > last)
            break;
    }
    __syncthreads();
    finish(last);
    if (live)
    {
#pragma unroll
        for (int j = 0; j < TILES; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                st[(int64_t) (16 * (wid + 4 * j) + 4 * g4 + i) * V + v] = S[j][i];
    }
}

// The walk of HGRN2 and Mamba-2, where what a chunk adds to the state does not hang on the state (u is there from the start): one workgroup per (entry, head, 16 columns of V), eight
// chunks between two barriers, D up to 128.  Wave w carries tile w of the state (16 rows) through the eight: K^T U of its rows, q S of its rows into LDS, S <- b S + K^T U; behind the barrier
// it sums chunk w's parts and finishes its rows.  The chain is a multiply-add per chunk, operands are asked for eight chunks ahead in the registers that they have just left, and a SIMD's two
// waves cover each other.  Bound by the operands' way to the CU (every 16 columns bring 16 KB of q and k a chunk: 17 - 20 bytes per clock) ahead of the MFMAs (68 of 32 clocks on four SIMDs a
// chunk): 1300 clocks a chunk.  Both launches, us, in brackets with chunk_walk_kernel: HGRN2 16 heads 128 x 128, 1021 rows 57 (69), Mamba-2 64 heads 128 x 64 57 (76).
// With four waves and a barrier per chunk (chunk_walk_kernel) a chunk's products, the barrier and the sums over the waves stood one after the
// other, 2100 clocks a chunk.  Tried on the way: a wave per chunk with all rows of the state, the state handed on through LDS (63 and 63; four waves 66 and 70: LDS and the fold beside idle MFMAs).
constexpr int SCAN = 8; // chunks at a time, waves
template <int DT, int MODE, int TILES>
__global__ __launch_bounds__(64 * SCAN) void eight_chunk_walk_kernel(const ChunkArgs a)
{
    static_assert(MODE != DELTA && TILES <= 2, "u hangs on the state; a wave per tile");
    constexpr int D = TILES * 64, NT = TILES * 4;
    extern __shared__ __attribute__((aligned(16))) float sm[];
    f32x4* part = reinterpret_cast<f32x4*>(sm);  // [2][8][NT][64] q S by turn, chunk, tile, lane
    f32x4* us = part + 2 * SCAN * NT * 64;       // [2][8][64] u by turn and chunk, SSM: dt_s f_{s+1} ... f_16 u
    const int e = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c16 = lane & 15, g4 = lane >> 4;
    const int v = blockIdx.z * 16 + c16, V = a.V, vc = v < V ? v : V - 1;
    const int first = a.ent_first[e], count = a.ent_count[e], last = (count + R - 1) / R - 1;
    if (last < 0)
        return;
    const int64_t slot0 = first / R + e;
    const int grp = MODE == SSM ? h / (a.heads / a.groups) : 0;
    const int tile = NT == SCAN ? wid : wid % NT; // (waves beyond the tiles go along; what they form is not used)
    float* st = a.state + (((int64_t) a.ent_slot[e] * a.heads + h) * D + 16 * tile + 4 * g4) * V + v;
    const bool live = v < V, carry = a.ent_pos0[e] > 0;

    f32x4 S;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        S[i] = live && carry ? st[(int64_t) i * V] : 0.f;
    const float dsk = MODE == SSM ? a.d_skip[h] : 0.f;

    typedef typename std::conditional<DT == DT_BF16, uint16_t, float>::type Raw;
    const Raw* vsrc = reinterpret_cast<const Raw*>(MODE == HGRN ? a.proj : a.xbc);
    const int64_t vld = MODE == HGRN ? a.ldp : a.ldx;
    const int64_t vcol = (MODE == HGRN ? 2 * a.heads * D : 0) + h * V + vc;
    f32x4 kt[SCAN], q[SCAN], b[SCAN], p, bt, ws; // by chunk, of this wave's tile; of this wave's chunk
    Raw vr[4], zr[4];
    auto row_of = [&](int j, int i) { return (int64_t) (first + min(j * R + 4 * g4 + i, count - 1)); };
    auto request_kt = [&](int c, int j) {
        const int64_t kg = MODE == SSM ? (slot0 + j) * a.groups + grp : (slot0 + j) * a.heads + h;
        kt[c] = *reinterpret_cast<const f32x4*>(a.kt + kg * D * R + (16 * tile + c16) * R + 4 * g4);
    };
    auto request_q = [&](int c, int j) {
        const int64_t ch = (slot0 + j) * a.heads + h, kg = MODE == SSM ? (slot0 + j) * a.groups + grp : ch;
        q[c] = *reinterpret_cast<const f32x4*>(a.qt + kg * R * D + c16 * D + 16 * tile + 4 * g4);
        if constexpr (MODE == SSM)
            b[c][0] = a.bc[ch * 48 + 2 * R];
        else
            b[c] = *reinterpret_cast<const f32x4*>(a.bc + ch * D + 16 * tile + 4 * g4);
    };
    auto leave_part = [&](int turn, int c, const f32x4& o) {
        if (NT == SCAN || wid < NT)
            part[((turn * SCAN + c) * NT + tile) * 64 + lane] = o;
    };
    auto request_u = [&](int j) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            vr[i] = vsrc[row_of(j, i) * vld + vcol];
        if constexpr (MODE == SSM)
            ws = *reinterpret_cast<const f32x4*>(a.bc + ((slot0 + j) * a.heads + h) * 48 + R + 4 * g4);
    };
    auto request_output = [&](int j) {
        const int64_t ch = (slot0 + j) * a.heads + h;
        p = *reinterpret_cast<const f32x4*>(a.pm + ch * R * R + c16 * R + 4 * g4);
        if constexpr (MODE == SSM)
        {
            bt = *reinterpret_cast<const f32x4*>(a.bc + ch * 48 + 4 * g4);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                zr[i] = reinterpret_cast<const Raw*>(a.proj)[row_of(j, i) * a.ldp + h * V + vc];
        }
    };
    auto cvt = [](Raw r) -> float {
        if constexpr (DT == DT_BF16)
            return bf2f(r);
        else
            return r;
    };
    // this wave's chunk's u, for all tiles
    auto leave_u = [&](int turn) {
        f32x4 u;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            u[i] = cvt(vr[i]);
        us[(turn * SCAN + wid) * 64 + lane] = MODE == SSM ? u * ws : u;
        return u;
    };

    request_u(min(wid, last));
    __builtin_amdgcn_sched_barrier(0); // (requests in the order in which they are used: the waits count them)
#pragma unroll
    for (int c = 0; c < SCAN; ++c)
    {
        if (c == 0)
            request_kt(0, 0);
        request_q(c, min(c, last));
        if (c + 1 < SCAN)
            request_kt(c + 1, min(c + 1, last));
        __builtin_amdgcn_sched_barrier(0);
    }
    request_output(min(wid, last));
    __builtin_amdgcn_sched_barrier(0);
    f32x4 u = leave_u(0);
    __syncthreads();
    for (int j0 = 0, turn = 0; j0 <= last; j0 += SCAN, turn ^= 1)
    {
        const int j = j0 + wid, next = min(j + SCAN, last); // (past the end the last chunk's operands, nothing of which counts)
        request_u(next);
        __builtin_amdgcn_sched_barrier(0);
        f32x4 uc[SCAN];
#pragma unroll
        for (int c = 0; c < SCAN; ++c)
            uc[c] = us[(turn * SCAN + c) * 64 + lane];
        // chunk c's q S beside chunk c + 1's K^T U: what S waits for was formed a chunk ahead
        f32x4 x = {0.f, 0.f, 0.f, 0.f}, o_before = x;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            x = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[0][i], uc[0][i], x, 0, 0, 0);
        request_kt(0, min(j0 + SCAN, last));
#pragma unroll
        for (int c = 0; c < SCAN; ++c)
        {
            f32x4 o = {0.f, 0.f, 0.f, 0.f}, x_next = o;
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                o = __builtin_amdgcn_mfma_f32_16x16x4f32(q[c][i], S[i], o, 0, 0, 0);
                if (c + 1 < SCAN)
                    x_next = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[c + 1][i], uc[c + 1][i], x_next, 0, 0, 0);
            }
            const f32x4 after = MODE == SSM ? S * b[c][0] + x : S * b[c] + x;
            S = j0 + c <= last ? after : S;
            if (c > 0)
                leave_part(turn, c - 1, o_before);
            x = x_next;
            o_before = o;
            __builtin_amdgcn_sched_barrier(0);
            const int after_j = min(j0 + SCAN + c, last);
            request_q(c, after_j);
            if (c + 1 < SCAN)
                request_kt(c + 1, min(j0 + SCAN + c + 1, last));
            __builtin_amdgcn_sched_barrier(0);
        }
        leave_part(turn, SCAN - 1, o_before);
        const f32x4 u_next = leave_u(turn ^ 1);
        __syncthreads();
        f32x4 past = part[(turn * SCAN + wid) * NT * 64 + lane];
#pragma unroll
        for (int n = 1; n < NT; ++n)
            past = past + part[((turn * SCAN + wid) * NT + n) * 64 + lane];
        if constexpr (MODE == SSM)
            past = past * bt;
        f32x4 y = past;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            y = __builtin_amdgcn_mfma_f32_16x16x4f32(p[i], u[i], y, 0, 0, 0);
        // the zeros of P above its diagonal meet every row: as in chunk_walk_kernel, a chunk with an infinity or a NaN row by row
        if (any_large(u))
            y = lower_product(p, u, 0, 4, past);
        if constexpr (MODE == SSM)
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                const float z = cvt(zr[i]);
                y[i] = fmaf(dsk, u[i], y[i]) * (z / (1.f + expf(-z)));
            }
        if (live && j <= last)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (j * R + 4 * g4 + i < count)
                    a.out[(int64_t) (first + j * R + 4 * g4 + i) * (a.heads * V) + h * V + v] = y[i];
        __builtin_amdgcn_sched_barrier(0);
        request_output(next);
        __builtin_amdgcn_sched_barrier(0);
        u = u_next;
    }
    if (live && wid < NT)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            st[(int64_t) i * V] = S[i];
}

inline int launched(const char* what)
{
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
    {
        set_error("%s launch failed: %s", what, hipGetErrorString(e));
        return -1;
    }
    return 0;
}

// Whether a step's walk is eight_chunk_walk_kernel.  Its turns are of eight chunks, however few of them an entry has left, and its LDS leaves room for one workgroup of D = 128 on a CU or two
// of 64, where chunk_walk_kernel's keep each other's waits covered: it is for entries that fill their turns, in no more workgroups than CUs.  Both launches by it, chunk_walk_kernel's as 1, bf16,
// longest entry of 7 / 8 / 9 / 13 / 14 / 16 / 17 / 19 / 24 / 25 / 32 / 64 chunks:
//   D 128, up to one workgroup a CU  HGRN2 1.02 / .99 / 1.12 / .99 / .96 / .92 / 1.02 / .98 / .89 / .97 / .86 / .84   Mamba-2 1.00 / .97 / 1.08 / .96 / .93 / .90 / .97 / .93 / .84 / .91 / .81 / .74
//   D 128, up to two                 HGRN2 1.14 / 1.09 / 1.29 / 1.11 / 1.09 / 1.04 / 1.18 / 1.13 / 1.02 / 1.14 / 1.01 / .98   Mamba-2 1.10 / 1.06 / 1.25 / 1.09 / 1.05 / .99 / 1.13 / 1.07 / .95 / 1.06 / .93 / .88
//   D 64, up to one                  HGRN2 1.12 / 1.08 / 1.28 / 1.12 / 1.08 / 1.03 / 1.18 / 1.13 / 1.02 / 1.12 / .99 / .96   Mamba-2 1.08 / 1.06 / 1.21 / 1.08 / 1.06 / 1.01 / 1.13 / 1.08 / .98 / 1.07 / .95 / .90
//   more workgroups: D 128 up to 1.5, D 64 up to 1.9; a step of 512 rows beside 31 single ones 1.04 - 1.09 and 1.5 - 1.8
// (four and more full rounds of them for Mamba-2, 0.92 at best, are left to chunk_walk_kernel: three are 1.07 - 1.4.)
template <int MODE>
bool eight_chunks_serve(const ChunkArgs& a)
{
    const int64_t wgs = (int64_t) a.entries * a.heads * ((a.V + 15) / 16), cus = launch_util::device_cus();
    const int chunks = (a.max_count + R - 1) / R, turns = (chunks + SCAN - 1) / SCAN;
    if (MODE == DELTA || a.D > 128)
        return false;
    if (a.D == 128 && wgs <= cus)
        return chunks >= 6 * turns + 2;
    const bool full = 15 * turns <= 2 * chunks; // 7.5 chunks a turn
    return MODE == SSM ? full && chunks >= 24 && wgs <= (a.D == 128 ? 2 : 1) * cus : full && chunks >= 46 && a.D == 64 && wgs <= cus;
}

template <int DT, int MODE>
void walk(const ChunkArgs& a, hipStream_t stream)
{
    const dim3 grid(a.entries, a.heads, (a.V + 15) / 16);
    if constexpr (MODE != DELTA)
        if (eight_chunks_serve<MODE>(a))
        {
            const auto kernel = a.D == 64 ? eight_chunk_walk_kernel<DT, MODE, 1> : eight_chunk_walk_kernel<DT, MODE, 2>;
            const size_t lds = sizeof(f32x4) * 2 * SCAN * 64 * ((size_t) a.D / 16 + 1);
            launch_util::ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), lds);
            hipLaunchKernelGGL(kernel, grid, dim3(64 * SCAN), lds, stream, a);
            return;
        }
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, a); };
    if constexpr (MODE == DELTA)
        switch (a.D / 64)
        {
        case 1: return go(delta_chunk_walk_kernel<DT, 1>);
        case 2: return go(delta_chunk_walk_kernel<DT, 2>);
        case 3: return go(delta_chunk_walk_kernel<DT, 3>);
        default: return go(delta_chunk_walk_kernel<DT, 4>);
        }
    else
        switch (a.D / 64)
        {
        case 1: return go(chunk_walk_kernel<DT, MODE, 1>);
        case 2: return go(chunk_walk_kernel<DT, MODE, 2>);
        case 3: return go(chunk_walk_kernel<DT, MODE, 3>);
        default: return go(chunk_walk_kernel<DT, MODE, 4>);
        }
}

template <int DT, int MODE>
int run(const ChunkArgs& a, hipStream_t stream)
{
    if constexpr (MODE == SSM)
    {
        const size_t lds = sizeof(float) * ((size_t) 2 * R * (a.D + 4) + 2 * (size_t) (a.heads / a.groups) * R);
        hipLaunchKernelGGL((ssm_prepare_kernel<DT>), dim3(a.slots, a.groups), dim3(256), lds, stream, a);
    }
    else
    {
        const size_t lds = sizeof(float) * ((size_t) 3 * R * a.D + R * R + R);
        hipLaunchKernelGGL((chunk_prepare_kernel<DT, MODE>), dim3(a.slots, a.heads), dim3(256), lds, stream, a);
    }
    walk<DT, MODE>(a, stream);
    return launched("stack_chunk");
}

// Lays the scratch of a step out in ws -> the floats it takes (ws null: only that)
size_t carve(ChunkArgs& a, int mode, int tokens, float* ws)
{
    a.slots = stack_chunk_slots(tokens, a.entries);
    const size_t c = a.slots, hd = (size_t) a.heads * a.D, vectors = mode == SSM ? (size_t) a.groups * a.D : hd;
    size_t at = 0;
    auto take = [&](size_t n) {
        float* p = ws ? ws + at : nullptr;
        at += n;
        return p;
    };
    a.qt = take(c * vectors * R);
    if (mode == DELTA)
        a.kb = take(c * hd * R);
    a.kt = take(c * vectors * R);
    a.pm = take(c * a.heads * R * R);
    if (mode == DELTA)
        a.tm = take(c * a.heads * R * R);
    a.bc = take(c * (mode == SSM ? (size_t) a.heads * 48 : hd));
    return at;
}

} // namespace

size_t stack_chunk_floats(StackChunkKind kind, int32_t tokens, int32_t entries, int32_t heads, int32_t groups, int32_t dim)
{
    ChunkArgs a;
    a.heads = heads;
    a.groups = groups;
    a.D = dim;
    a.entries = entries;
    return carve(a, kind, tokens, nullptr);
}

bool stack_chunk_serves(int32_t dim, int32_t max_count)
{
    // from two chunks on: a portion of 32 rows takes 32 us row by row
    return dim % 64 == 0 && dim >= 64 && dim <= 256 && max_count >= 2 * R;
}

int launch_stack_chunk_hgrn2(const StackHgrnParams& p, hipStream_t stream)
{
    ChunkArgs a;
    a.heads = p.heads;
    a.D = p.dim;
    a.V = p.vdim;
    a.entries = p.entries;
    a.max_count = p.max_count;
    a.proj = p.proj;
    a.ldp = p.ldp;
    a.f_bias = p.f_bias;
    a.lower = p.lower;
    a.state = p.state;
    a.out = p.o32;
    a.ent_slot = p.ent_slot;
    a.ent_first = p.ent_first;
    a.ent_count = p.ent_count;
    a.ent_pos0 = p.ent_pos0;
    if (!stack_chunk_serves(p.dim, p.max_count) || !p.chunk_ws || carve(a, HGRN, p.tokens, p.chunk_ws) > p.chunk_floats)
        return 1;
    return p.dtype == DT_BF16 ? run<DT_BF16, HGRN>(a, stream) : run<DT_FLOAT, HGRN>(a, stream);
}

int launch_stack_chunk_delta(const StackDeltaParams& p, hipStream_t stream)
{
    ChunkArgs a;
    a.heads = p.heads;
    a.qk_heads = p.qk_heads;
    a.D = p.dim;
    a.V = p.vdim;
    a.entries = p.entries;
    a.max_count = p.max_count;
    a.xbc = p.x;
    a.ldx = 2 * (int64_t) p.qk_heads * p.dim + (int64_t) p.heads * p.vdim;
    a.decay_raw = p.decay_raw;
    a.dt_bias = p.dt_bias;
    a.a_log = p.a_log;
    a.beta_raw = p.beta_raw;
    a.ld_beta = p.ld_beta;
    a.state = p.state;
    a.out = p.o32;
    a.ent_slot = p.ent_slot;
    a.ent_first = p.ent_first;
    a.ent_count = p.ent_count;
    a.ent_pos0 = p.ent_pos0;
    if (!stack_chunk_serves(p.dim, p.max_count) || !p.chunk_ws || carve(a, DELTA, p.tokens, p.chunk_ws) > p.chunk_floats)
        return 1;
    return p.dtype == DT_BF16 ? run<DT_BF16, DELTA>(a, stream) : run<DT_FLOAT, DELTA>(a, stream);
}

int launch_stack_chunk_ssm(const StackSsmParams& p, hipStream_t stream)
{
    ChunkArgs a;
    a.heads = p.heads;
    a.groups = p.groups;
    a.D = p.state;
    a.V = p.vdim;
    a.entries = p.entries;
    a.max_count = p.max_count;
    a.proj = p.proj;
    a.ldp = p.ldp;
    a.xbc = p.xbc;
    a.ldx = (int64_t) p.heads * p.vdim + 2 * (int64_t) p.groups * p.state;
    a.dt_bias = p.dt_bias;
    a.a_log = p.a_log;
    a.d_skip = p.d_skip;
    a.state = p.ssm_state;
    a.out = p.y32;
    a.ent_slot = p.ent_slot;
    a.ent_first = p.ent_first;
    a.ent_count = p.ent_count;
    a.ent_pos0 = p.ent_pos0;
    // (the heads of a group share a workgroup's LDS in the first launch)
    if (!stack_chunk_serves(p.state, p.max_count) || p.heads / p.groups > 128 || !p.chunk_ws || carve(a, SSM, p.tokens, p.chunk_ws) > p.chunk_floats)
        return 1;
    return p.dtype == DT_BF16 ? run<DT_BF16, SSM>(a, stream) : run<DT_FLOAT, SSM>(a, stream);
}

} // namespace kernels
} // namespace tllm
