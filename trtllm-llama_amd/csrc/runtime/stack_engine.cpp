// extern "C" surface of include/tllm_stack_api.h: the ragged-batch step executor for run-time described decoder stacks.
//
// One step = embedding -> the layer runs in order -> final norm + head on the wanted rows -> arg-max.  A layer run is
//   h1, h2 = norm1(x), norm2(x)                                  one launch (the two norms share the normalised row)
//   P1 = h1 [Wq; Wk; Wv; Wrg1]^T   (hgrn2: [Wq; Wf; Wv; Wrg1])    one product: everything that reads h1
//   ctx = mixer(P1)                                              rotary + cache append + attention | recurrence + head norm
//   x += sigmoid(P1[rg1] + b1) * (ctx Wo^T)                      product with the gated-residual seam in its epilogue
//   a = gelu(h2 Wgate^T) * (h2 Wup^T), rg2 = h2 Wrg2^T             one product: gate and up rows in turn, the gating in its epilogue
//   x += sigmoid(rg2 + b2) * (a Wdown^T)
// on the packed rows of the step (block=parallel, residual=gated).  With block=sequential, residual=hyper a layer run is pre-norm
// with `streams` hyper-connected copies of the residual:
//   h1 = norm1(sum_s in1[s] x_s)                                  one launch, which also lands the sublayer before it (below)
//   P1 = h1 [Wq; Wk; Wv; Wg]^T  (latent attention: [Wq; Wdkv])    mixer as above, per-head output gate inside the attention launch
//   y = ctx Wo^T (fp32);  x_t <- sum_s mix1[s, t] x_s + out1[t] y   folded into the next launch that reads the streams
//   h2 = norm2(sum_s in2[s] x_s);  a = relu(h2 Wup^T)^2 (product epilogue);  y = a Wdown^T;  x_t <- sum_s mix2[s, t] x_s + out2[t] y
// A mamba2 mixer is  P1 = h1 W_in^T = [z | x | B | C | dt]  ->  convolution + silu of x | B | C (and the sequence's new tail)  ->  the
// recurrence with skip and gate  ->  RMS norm in parts of the row;  a latent layer with a query latent projects [W_dq; W_dkv], norms
// the query latent and expands it before the latent's pointwise part.  A routed feed-forward is  router (fp32 logits, softmax, kept
// groups, top-k)  ->  (token, expert) pairs ordered by expert  ->  grouped product with silu(gate) * up in its epilogue  ->  down_e
// grouped product in fp32  ->  weighted sum per token (identity experts add w h).  With block=parallel, residual=plain a layer run has
// ONE norm that both sublayers read, and plain fp32 sums:
//   P = h [Wq; Wdkv; Wg | Wshared_up | Wrouter]^T                 one product, three output sections: the mixer's columns, the shared
//                                                                 expert's relu^2 activations (behind the context row), fp32 router logits
//   mixer (the per-head output gate inside the attention launch)  -> ctx
//   x += [ctx | a_shared] [Wo | Wshared_down]^T                   one product: the two sublayers' plain parts
//   routed experts as above, read through the token of each slot; x += sum_k w_k y_k
//   side: g = gelu(Wgate x) * e (epilogue: the layer's part of the token's side embedding); y = Wproj g
//   x += norm(y); x += the next pass's step; h = norm1(x)         one launch, which also starts the next layer
// With block=sequential, residual=plain the sublayers of the hyper form run on one plain sum, landed by that last launch:
//   x += m norm1b(y); h = norm2(x)                                one launch between two sublayers (norm2b / norm1 behind the second)
//   P = h [Wshared gate, up rows in turn | Wrouter; Wsg]^T        one product: the shared expert's activations, fp32 logits and gate
//   shared down -> y; experts as above; y = sigmoid(z_sg) y + sum_k w_k y_k
// A layer with weights_of runs on another layer's
// device tensors; caches and states belong to runs.
// The residual streams are fp32 in both element types.
#include "../../../include/tllm_stack_api.h"
#include "../kernels/stack_kernels.h"
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <chrono>
#include <cstring>
#include <map>
#include <string>
#include <vector>

using namespace tllm;
using namespace tllm::kernels;

namespace
{

struct HostTensor
{
    std::vector<int64_t> dims;
    std::vector<float> v; // every weight passes through fp32 on the host (bfloat16 -> fp32 is exact)
    int64_t numel() const
    {
        int64_t n = 1;
        for (auto d : dims)
            n *= d;
        return n;
    }
};

enum MixerKind
{
    MIX_ATTENTION = 0,
    MIX_HGRN2 = 1,
    MIX_LATENT = 2,
    MIX_MAMBA2 = 3,
    MIX_DELTA = 4
};
enum MlpKind
{
    MLP_GELU_GATE = 0, // W_down (gelu_tanh(W_gate h) * W_up h)
    MLP_RELU2 = 1,     // W_down relu(W_up h)^2
    MLP_MOE = 2        // routed experts of size ff - W_down (silu(W_gate h) * W_up h) or W_down relu(W_up h)^2 -, the last `identity` router
                       // outputs return h; optionally a shared expert of size shared_ff that every token uses
};
constexpr int kSideParts = 16; // the token input's gate product has few columns: room for this many parts of its K

struct HyperW
{
    float *mix = nullptr, *out = nullptr, *in = nullptr;
};

struct Layer
{
    int kind = MIX_ATTENTION;
    int heads = 0, kv_heads = 0, dim = 0, vdim = 0, maps = 1, ff = 0, head_norm = 0;
    double diff = 0, scale = 1, softcap = 0;
    int rot_dims = 0;
    double rot_base = 10000, rot_factor = 0, rot_original = 0, rot_fast = 0, rot_slow = 0, rot_low = 1, rot_high = 4;
    // derived
    int n_q = 0, n_k = 0, n_v = 0, n_mix = 0, n_ctx = 0; // columns of P1: q | k (or f) | v | rg1
    float lambda = 0.f, mscale = 1.f;
    int mlp = MLP_GELU_GATE;
    int qkv_bias = 0, qk_norm = 0, head_temp = 0, pos_bias = 0 /* 0 none, 1 linear, 2 log */, mask = MASK_CAUSAL, mask_size = 0,
        weights = WEIGHTS_SOFTMAX, sink = 0, out_gate = 0;
    double slope_base = 8;
    int kv_rank = 0, rot_part = 0;  // latent attention: rank of the latent, size of the shared rotated key part (rot_dims of it turn)
    int n_gate = 0, n_rg = 0;       // further columns of P1: per-head output gates, the gated residual's projection
    int n_lat = 0;                  // latent attention: heads * kv_rank
    int q_rank = 0, rot_halves = 0; // latent attention: rank of a query latent (0: queries straight from the input), half-split pairs
    int weights_of = -1;            // the layer whose weights this one runs on (its cache / state is its own)
    int groups = 1, taps = 0, ssm_norm_groups = 1, n_conv = 0; // mamba2 (dim = state rows): B / C groups, convolution taps, parts of the output norm
    int experts = 0, identity = 0, top = 0, route_groups = 1, route_keep = 1; // moe
    double route_scale = 1;
    int expert_relu2 = 0, route_norm = 0, shared_ff = 0, n_route = 0, n_pad = 0; // moe: experts of the relu^2 form, weights divided by their sum; columns of P
    int route_bias = 0, shared_gate = 0, n_shared = 0; // moe: biased router logits; a sigmoid gate per token on the shared expert; columns of its first product
    int rot_linear = 0, v_mix = 0;                     // attention: frequencies divided by rot_factor; values mixed with those of the first layer that mixes
    float vmix = 0.f;
    int route_sigmoid = 0, route_weight_input = 0; // moe: sigmoid scores instead of a softmax; the weight scales the expert's input
    int mask_keep = 0, talk = 0, values_are_keys = 0, gate_wide = 0, qk_norm_weight = 0, o_bias = 0, rot_banded = 0; // attention
    int decay_rank = 0, gate_rank = 0, n_beta = 0; // delta_rule: ranks of the two low-rank projections, padded beta columns
    // device
    void *w_mix = nullptr, *w_o = nullptr, *w_gu = nullptr, *w_down = nullptr, *w_ukT = nullptr, *w_uv = nullptr;
    float *norm1 = nullptr, *norm2 = nullptr, *norm1b = nullptr, *norm2b = nullptr, *route_b = nullptr, *rg1_b = nullptr, *rg2_b = nullptr, *f_bias = nullptr, *lower = nullptr, *hnorm = nullptr,
          *freq = nullptr, *bias = nullptr, *temp = nullptr, *slope = nullptr, *r1 = nullptr, *r2 = nullptr, *sinkv = nullptr, *wbias = nullptr,
          *lat_norm = nullptr, *cq_norm = nullptr, *conv_w = nullptr, *conv_b = nullptr, *dt_bias = nullptr, *a_log = nullptr,
          *d_skip = nullptr, *router_w = nullptr, *correction = nullptr, *talkw = nullptr, *q_norm = nullptr, *k_norm = nullptr, *o_biasv = nullptr,
          *shift = nullptr;
    void *w_a2 = nullptr, *w_g2 = nullptr; // delta_rule: the second halves of the decay's and the gate's low-rank projections
    bool low_pair = false;                 // ... of one shape: both in w_a2, one product of two where one launch serves it
    void* w_uq = nullptr;
    void *w_shared_up = nullptr, *w_shared_down = nullptr; // shared expert (where it is not part of w_mix / w_o)
    void *side_gate = nullptr, *side_proj = nullptr;       // per-layer token input
    float* side_norm = nullptr;
    HyperW hc[2];
};

struct Run
{
    int layer = 0, pass = 0;
    bool enters_pass = false;
    void *k_pool = nullptr, *v_pool = nullptr; // attention
    float* state = nullptr;                    // hgrn2, mamba2
    float* conv_state = nullptr;               // mamba2, delta_rule: the last inputs of the convolution, in a ring of taps rows (fed)
    float* shift_carry = nullptr;              // token shift: the sequence's last normed row, [slots, width]
};

// Rows go on to the caller as they land in pinned memory, while those behind them are still on their way, and without the runtime's wait for the end of the stream: a marker
// behind the last launch, the wait for it and its wake-up took 12 - 30 us a step (a step of one row of 32000: 329 us with it, 317; eight rows 567, 545).  -> how many of the
// rows: the wait ends after SPIN, a core's time, behind which the runtime's own counts for little; a step whose products alone last that long does without (lands_soon).
//
// What may follow, on whichever stream: a part's choice is stored behind a release at system scope, by the last launch of its step, so that all which that stream ran
// before comes ahead of the host's acquire here, and of what the host launches from then on.  Left of the step is the end of a launch that has read and written all it will.
// (So no event behind every step, a marker in the streams of all for the few who change theirs.)
constexpr auto SPIN = std::chrono::milliseconds(2);
int copy_as_they_land(float* to, const float* landing, const StackChoice* choice, int rows, int vocab)
{
    const int parts = stack_choice_parts(vocab);
    const auto until = std::chrono::steady_clock::now() + SPIN;
    for (int r = 0; r < rows; ++r)
    {
        for (int i = 0; i < parts; ++i)
            for (int tries = 0; __atomic_load_n(&choice[(size_t) r * parts + i].at, __ATOMIC_ACQUIRE) == stack_no_choice.at;)
            {
                if (++tries % 64 == 0 && std::chrono::steady_clock::now() > until)
                    return r;
                __builtin_ia32_pause();
            }
        if (to)
            std::memcpy(to + (size_t) r * vocab, landing + (size_t) r * vocab, (size_t) vocab * 4);
    }
    return rows;
}

// The caller's rows are mostly memory that the system has yet to give: their pages come in while the GPU works, with what they hold unchanged,
// instead of behind it.
void bring_in(float* rows, size_t bytes)
{
    volatile char* p = reinterpret_cast<volatile char*>(rows);
    for (size_t at = 0; at < bytes; at += 4096)
        p[at] = p[at];
    p[bytes - 1] = p[bytes - 1];
}

} // namespace

struct tllm_stack
{
    std::map<std::string, std::string> cfg;
    std::map<std::string, HostTensor> host;
    int dtype = DT_BF16, es = 2;
    int width = 0, vocab = 0, groups = 1, page = 64, blocks = 0, slots = 0, taps = 0;
    int loop_start = 0, loop_stop = 0, loop_times = 1;
    bool sequential = false, hyper = false, plain = false;
    bool side_by_side = false; // a plain residual whose sublayers read one normed row
    int embed_norm = 0, loop_input = 1, side_dim = 0, post_norm = 0, tied_head = 0;
    int v_mix_first = -1, v_mix_cols = 0; // the first layer that mixes values, and how many values a token has there
    float resid_mult = 1.f;
    void* v_first = nullptr;   // [tokens, v_mix_cols]: that layer's values of the step's tokens
    float* shared_z = nullptr; // [tokens]: the shared expert's gate ahead of its sigmoid
    float logit_scale = 1.f, logit_cap = 0.f;
    void *side_embed = nullptr, *x_el = nullptr, *side_act = nullptr, *act_sh = nullptr;
    float *embed_norm_w = nullptr, *route_z = nullptr, *split_ws = nullptr;
    int streams = 1;
    float norm_offset = 0.f, *ones = nullptr;
    float eps = 1e-5f, emb_scale = 1.f;
    std::vector<Layer> layers;
    std::vector<Run> runs;
    void *embed = nullptr, *head = nullptr;
    float *final_norm = nullptr, *loop_step = nullptr, *attn_ws = nullptr;
    bool finalized = false;
    int64_t weight_bytes = 0;
    double token_flops = 0; // of a token's products, without the head's
    std::vector<void*> owned;
    // scratch, grown to the largest step seen
    int cap_tokens = 0, cap_want = 0, cap_ints = 0;
    float* chunk_ws = nullptr; // scratch of the chunked recurrences
    size_t chunk_floats = 0;
    float *x = nullptr, *x0 = nullptr, *o32 = nullptr, *logits = nullptr, *tap = nullptr, *y32 = nullptr;
    void *h1 = nullptr, *h2 = nullptr, *proj = nullptr, *q = nullptr, *ctx = nullptr, *act = nullptr, *hw = nullptr, *lat = nullptr;
    int32_t *ints = nullptr, *ids_out = nullptr, *pinned = nullptr;
    // pinned host memory that a few wanted rows are delivered to: the parts' choices, then the logits
    StackChoice* land_choice = nullptr;
    float* land_rows = nullptr;
    int land_cap = 0; // rows
    void *xbc = nullptr, *cq = nullptr, *qfull = nullptr, *moe_a = nullptr;
    float *moe_y = nullptr, *moe_w = nullptr;
    int32_t* moe_i = nullptr;
    uint32_t* moe_ticket = nullptr; // behind moe_i's values: zero between launches
    // pair embedding (a hashed row per (previous token, token)) and token shift; the previous token of every slot's sequence
    int pair_buckets = 0, pair_mul_prev = 0, pair_mul_cur = 0, token_shift = 0;
    void* pair_table = nullptr;
    std::vector<int32_t> last_tok;
    std::vector<int32_t> fed; // rows that every slot's sequence has had: where its convolutions' rings of raw inputs stand, whatever positions the caller counts
    float *h32 = nullptr, *dl_a = nullptr, *dl_g = nullptr;
    void* pairs = nullptr; // talking heads: every query head's weights over every value head's rows, [tokens, heads * kv_heads * vdim]
    int max_hd = 0, max_pairs = 0, max_sh = 0;
    int max_proj = 0, max_q = 0, max_ctx = 0, max_ff = 0, max_lat = 0, max_conv = 0, max_qrank = 0, max_qfull = 0, max_top = 0, max_experts = 0, max_outputs = 0;
    int tap_tokens = 0;

    ~tllm_stack()
    {
        for (void* p : owned)
            (void) hipFree(p);
        free_scratch();
        if (pinned)
            (void) hipHostFree(pinned);
        if (land_choice)
            (void) hipHostFree(land_choice);
    }
    void free_scratch()
    {
        void* all[] = {chunk_ws, v_first, shared_z, split_ws, x_el, side_act, act_sh, route_z, x, x0, o32, logits, tap, y32, h1, h2, proj, q, ctx, act, hw, lat, ints, ids_out, xbc, cq, qfull, moe_a, moe_y, moe_w, moe_i,
            h32, dl_a, pairs};
        for (void* p : all)
            if (p)
                (void) hipFree(p);
        x_el = side_act = act_sh = nullptr;
        v_first = nullptr;
        route_z = split_ws = shared_z = chunk_ws = nullptr;
        chunk_floats = 0;
        x = x0 = o32 = logits = tap = y32 = nullptr;
        h1 = h2 = proj = q = ctx = act = hw = lat = nullptr;
        ints = ids_out = nullptr;
        xbc = cq = qfull = moe_a = nullptr;
        moe_y = moe_w = nullptr;
        moe_i = nullptr;
        moe_ticket = nullptr;
        h32 = dl_a = dl_g = nullptr;
        pairs = nullptr;
    }
};

namespace
{

#define HIP_OK(call)                                                                                                              \
    do                                                                                                                              \
    {                                                                                                                               \
        const hipError_t e_ = (call);                                                                                               \
        if (e_ != hipSuccess)                                                                                                       \
        {                                                                                                                           \
            (void) hipGetLastError(); /* reported here: the next launch's check must not find it */                                \
            set_error("stack engine: %s failed: %s", #call, hipGetErrorString(e_));                                               \
            return -1;                                                                                                              \
        }                                                                                                                           \
    } while (0)

inline uint16_t host_f2bf(float f)
{
    uint32_t u;
    std::memcpy(&u, &f, 4);
    if ((u & 0x7fffffffu) > 0x7f800000u)
        return (uint16_t) ((u >> 16) | 0x40u);
    return (uint16_t) ((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

double getd(const tllm_stack* s, const std::string& k, double dflt)
{
    auto it = s->cfg.find(k);
    return it == s->cfg.end() ? dflt : std::atof(it->second.c_str());
}
int geti(const tllm_stack* s, const std::string& k, int dflt)
{
    auto it = s->cfg.find(k);
    return it == s->cfg.end() ? dflt : std::atoi(it->second.c_str());
}
std::string gets(const tllm_stack* s, const std::string& k, const std::string& dflt)
{
    auto it = s->cfg.find(k);
    return it == s->cfg.end() ? dflt : it->second;
}

// rows of several [n_i, K] host matrices stacked into one device matrix of the engine's element type
int upload_rows(tllm_stack* s, const std::vector<const HostTensor*>& parts, void** out)
{
    int64_t n = 0;
    for (auto* t : parts)
        n += t->numel();
    void* d = nullptr;
    HIP_OK(hipMalloc(&d, (size_t) (n ? n : 1) * s->es));
    s->owned.push_back(d);
    s->weight_bytes += n * s->es;
    int64_t off = 0;
    std::vector<uint16_t> tmp;
    for (auto* t : parts)
    {
        if (s->dtype == DT_FLOAT)
            HIP_OK(hipMemcpy((char*) d + off * 4, t->v.data(), t->v.size() * 4, hipMemcpyHostToDevice));
        else
        {
            tmp.resize(t->v.size());
            for (size_t i = 0; i < tmp.size(); ++i)
                tmp[i] = host_f2bf(t->v[i]);
            HIP_OK(hipMemcpy((char*) d + off * 2, tmp.data(), tmp.size() * 2, hipMemcpyHostToDevice));
        }
        off += t->numel();
    }
    *out = d;
    return 0;
}

const HostTensor* need(tllm_stack* s, const std::string& name, std::initializer_list<int64_t> dims);

// A gate's and a gated matrix ([n, K] each) with their rows alternating, as the products' gate activations want them; takes the place of the
// gate's host tensor (neither is used again)
const HostTensor* need_gated(tllm_stack* s, const std::string& gate, const std::string& up, int64_t n, int64_t K)
{
    if (!need(s, gate, {n, K}) || !need(s, up, {n, K}))
        return nullptr;
    HostTensor &g = s->host[gate], &u = s->host[up];
    std::vector<float> both((size_t) (2 * n * K));
    for (int64_t r = 0; r < n; ++r)
    {
        std::copy_n(g.v.data() + r * K, K, both.data() + 2 * r * K);
        std::copy_n(u.v.data() + r * K, K, both.data() + (2 * r + 1) * K);
    }
    g.v.swap(both);
    g.dims = {2 * n, K};
    u.v.clear();
    return &g;
}

int upload_f32(tllm_stack* s, const float* v, size_t n, float** out)
{
    void* d = nullptr;
    HIP_OK(hipMalloc(&d, (n ? n : 1) * 4));
    s->owned.push_back(d);
    s->weight_bytes += (int64_t) n * 4;
    HIP_OK(hipMemcpy(d, v, n * 4, hipMemcpyHostToDevice));
    *out = (float*) d;
    return 0;
}

const HostTensor* need(tllm_stack* s, const std::string& name, std::initializer_list<int64_t> dims)
{
    auto it = s->host.find(name);
    if (it == s->host.end())
    {
        set_error("tllm_stack_finalize: tensor %s is missing", name.c_str());
        return nullptr;
    }
    const std::vector<int64_t> want(dims);
    if (it->second.dims != want)
    {
        std::string have, w;
        for (auto d : it->second.dims)
            have += std::to_string(d) + " ";
        for (auto d : want)
            w += std::to_string(d) + " ";
        set_error("tllm_stack_finalize: tensor %s has shape [ %s], the configuration asks for [ %s]", name.c_str(), have.c_str(), w.c_str());
        return nullptr;
    }
    return &it->second;
}

int alloc_zero(tllm_stack* s, size_t bytes, void** out)
{
    void* d = nullptr;
    HIP_OK(hipMalloc(&d, bytes ? bytes : 16));
    s->owned.push_back(d);
    HIP_OK(hipMemset(d, 0, bytes ? bytes : 16));
    *out = d;
    return 0;
}

// Room in pinned host memory for a step's wanted rows, if they are few: -> whether they are delivered there.  kLandBytes bounds what an engine
// pins; beyond it the rows go to the caller's memory by copy commands.  A step of one small layer with 1 / 8 / 64 wanted rows of 32000
// values, us: 85 / 139 / 534 delivered, 135 / 186 / 632 by commands.
constexpr size_t kLandBytes = 8 << 20;
bool ensure_landing(tllm_stack* s, int want)
{
    const size_t row = (size_t) s->vocab * 4, parts = (size_t) stack_choice_parts(s->vocab);
    if (want < 1 || row * want > kLandBytes || want > 65535) // (a row is a workgroup row of the launch)
        return false;
    if (want <= s->land_cap)
        return true;
    if (s->land_choice)
    {
        (void) hipDeviceSynchronize(); // (a step that ended in an error may still be under way)
        (void) hipHostFree(s->land_choice);
    }
    // (twice the rows at least: as requests come in one by one, few of their steps pin anew)
    const size_t rows = std::min(kLandBytes / row, std::max((size_t) want, 2 * (size_t) s->land_cap));
    s->land_choice = nullptr;
    s->land_cap = 0;
    const size_t head = (sizeof(StackChoice) * parts * rows + 63) / 64 * 64;
    void* m = nullptr;
    if (hipHostMalloc(&m, head + row * rows, hipHostMallocDefault) != hipSuccess)
    {
        (void) hipGetLastError();
        return false;
    }
    s->land_choice = (StackChoice*) m;
    s->land_rows = (float*) ((char*) m + head);
    s->land_cap = (int) rows;
    return true;
}

// Whether a step of `tokens` may end within SPIN: its products do at the quickest rates measured here, 1.31 PFLOP/s in bfloat16, 0.15 (the chip's) in plain fp32.
bool lands_soon(const tllm_stack* s, int tokens)
{
    const double rate = s->dtype == DT_BF16 ? 1.31e15 : 0.15e15;
    return tokens * s->token_flops < rate * std::chrono::duration<double>(SPIN).count();
}

int ensure_scratch(tllm_stack* s, int tokens, int want, int n_ints)
{
    if (tokens > s->cap_tokens || want > s->cap_want || n_ints > s->cap_ints)
    {
        HIP_OK(hipDeviceSynchronize());
        s->free_scratch();
        if (s->pinned)
        {
            (void) hipHostFree(s->pinned);
            s->pinned = nullptr;
        }
        const size_t T = (size_t) std::max(tokens, s->cap_tokens), W = (size_t) std::max(want, s->cap_want);
        const size_t NI = (size_t) std::max(n_ints, s->cap_ints);
        s->cap_tokens = s->cap_want = s->cap_ints = 0; // (nothing is there until all of it is)
        const size_t es = s->es, wd = s->width;
        HIP_OK(hipMalloc((void**) &s->x, T * wd * 4 * (size_t) s->streams));
        HIP_OK(hipMalloc((void**) &s->y32, T * wd * 4));
        HIP_OK(hipMalloc(&s->lat, T * std::max(s->max_lat, 1) * es));
        HIP_OK(hipMalloc((void**) &s->x0, T * wd * 4));
        HIP_OK(hipMalloc((void**) &s->o32, T * std::max(s->max_ctx, 1) * 4));
        HIP_OK(hipMalloc((void**) &s->logits, W * s->vocab * 4));
        HIP_OK(hipMalloc(&s->h1, T * wd * es));
        HIP_OK(hipMalloc(&s->h2, T * wd * es));
        HIP_OK(hipMalloc(&s->proj, T * std::max(s->max_proj, 1) * es));
        HIP_OK(hipMalloc(&s->q, T * std::max(s->max_q, 1) * es));
        HIP_OK(hipMalloc(&s->ctx, T * std::max(s->max_ctx, 1) * es));
        HIP_OK(hipMalloc(&s->act, T * std::max(s->max_ff, 1) * es));
        HIP_OK(hipMalloc(&s->x_el, (s->side_dim ? T * wd : 1) * es));
        HIP_OK(hipMalloc(&s->act_sh, T * std::max(s->max_sh, 1) * es));
        HIP_OK(hipMalloc((void**) &s->route_z, (s->plain ? T * std::max(s->max_outputs, 1) : 1) * 4));
        HIP_OK(hipMalloc((void**) &s->shared_z, T * 4));
        HIP_OK(hipMalloc(&s->v_first, T * std::max(s->v_mix_cols, 1) * es));
        HIP_OK(hipMalloc((void**) &s->split_ws, T * (size_t) std::max(s->side_dim, 1) * kSideParts * 4));
        HIP_OK(hipMalloc(&s->side_act, T * std::max(s->side_dim, 1) * es));
        HIP_OK(hipMalloc(&s->hw, W * wd * es));
        HIP_OK(hipMalloc((void**) &s->ints, NI * 4));
        HIP_OK(hipMalloc((void**) &s->ids_out, W * 4));
        HIP_OK(hipMalloc(&s->xbc, T * std::max(s->max_conv, 1) * es));
        HIP_OK(hipMalloc(&s->cq, T * std::max(s->max_qrank, 1) * es));
        HIP_OK(hipMalloc(&s->qfull, T * std::max(s->max_qfull, 1) * es));
        HIP_OK(hipMalloc((void**) &s->h32, (s->token_shift ? T * wd : 1) * 4));
        HIP_OK(hipMalloc(&s->pairs, T * std::max(s->max_pairs, 1) * es));
        const size_t n_a = (T * std::max(s->max_hd, 1) + 63) / 64 * 64;
        HIP_OK(hipMalloc((void**) &s->dl_a, (n_a + (s->max_hd ? T * std::max(s->max_ctx, 1) : 1)) * 4)); // one block: a product of two writes both
        s->dl_g = s->dl_a + n_a;
        {
            // a mixture of experts works on one row per (token, chosen expert)
            const size_t pairs = T * (size_t) std::max(s->max_top, 1);
            HIP_OK(hipMalloc(&s->moe_a, (s->max_top ? pairs * wd : 1) * es));
            HIP_OK(hipMalloc((void**) &s->moe_y, (s->max_top ? pairs * wd : 1) * 4));
            HIP_OK(hipMalloc((void**) &s->moe_w, (pairs + T * (size_t) (s->max_outputs + 1)) * 4));
            const size_t n_moe_i = 4 * pairs + (size_t) s->max_experts + 1;
            HIP_OK(hipMalloc((void**) &s->moe_i, (n_moe_i + 1) * 4));
            s->moe_ticket = (uint32_t*) s->moe_i + n_moe_i;
            const uint32_t none = 0;
            HIP_OK(hipMemcpy(s->moe_ticket, &none, sizeof(none), hipMemcpyHostToDevice));
        }
        HIP_OK(hipHostMalloc((void**) &s->pinned, NI * 4, hipHostMallocDefault));
        if (s->taps)
            HIP_OK(hipMalloc((void**) &s->tap, s->runs.size() * T * wd * 4));
        // last, since a step does without it: where there is no room for it, its rows go one by one
        for (const auto& l : s->layers)
            if ((l.kind == MIX_DELTA || l.kind == MIX_HGRN2 || l.kind == MIX_MAMBA2) && stack_chunk_serves(l.dim, (int) T))
                s->chunk_floats = std::max(s->chunk_floats, stack_chunk_floats(l.kind == MIX_DELTA ? CHUNK_DELTA : l.kind == MIX_HGRN2 ? CHUNK_HGRN2 : CHUNK_SSM,
                                                                (int) T, std::min((int) T, s->slots), l.heads, l.groups, l.dim));
        if (s->chunk_floats && hipMalloc((void**) &s->chunk_ws, s->chunk_floats * 4) != hipSuccess)
        {
            (void) hipGetLastError();
            s->chunk_ws = nullptr;
            s->chunk_floats = 0;
        }
        s->cap_tokens = (int) T;
        s->cap_want = (int) W;
        s->cap_ints = (int) NI;
    }
    return 0;
}

} // namespace

extern "C" {

tllm_stack_t tllm_stack_create(const char* config_text)
{
    if (!config_text)
    {
        set_error("tllm_stack_create: no configuration");
        return nullptr;
    }
    auto* s = new tllm_stack();
    std::string text(config_text);
    size_t at = 0;
    while (at < text.size())
    {
        size_t nl = text.find('\n', at);
        if (nl == std::string::npos)
            nl = text.size();
        const std::string line = text.substr(at, nl - at);
        at = nl + 1;
        const size_t eq = line.find('=');
        if (eq == std::string::npos)
            continue;
        s->cfg[line.substr(0, eq)] = line.substr(eq + 1);
    }
    const std::string dt = gets(s, "dtype", "bfloat16");
    if (dt == "bfloat16")
        s->dtype = DT_BF16, s->es = 2;
    else if (dt == "float32")
        s->dtype = DT_FLOAT, s->es = 4;
    else
    {
        set_error("tllm_stack_create: dtype %s (bfloat16 or float32)", dt.c_str());
        delete s;
        return nullptr;
    }
    s->width = geti(s, "width", 0);
    s->vocab = geti(s, "vocab", 0);
    s->groups = geti(s, "norm_groups", 1);
    s->eps = (float) getd(s, "norm_eps", 1e-5);
    s->emb_scale = (float) getd(s, "embedding_scale", 1.0);
    s->page = geti(s, "page_size", 64);
    s->blocks = geti(s, "num_blocks", 0);
    s->slots = geti(s, "num_slots", 0);
    s->taps = geti(s, "debug_taps", 0);
    s->loop_start = geti(s, "loop_start", 0);
    s->loop_stop = geti(s, "loop_stop", 0);
    s->loop_times = geti(s, "loop_times", 1);
    s->norm_offset = (float) getd(s, "norm_offset", 0.0);
    s->streams = geti(s, "streams", 1);
    s->pair_buckets = geti(s, "pair_buckets", 0);
    if (s->pair_buckets > 0)
    {
        // the multipliers only matter modulo the bucket count: (a m) mod B = (a (m mod B)) mod B, and the kernel's 64-bit products then
        // have room for any vocabulary
        auto mod_b = [&](const char* key) {
            const long long m = std::atoll(gets(s, key, "0").c_str()) % s->pair_buckets;
            return (int) (m < 0 ? m + s->pair_buckets : m);
        };
        s->pair_mul_prev = mod_b("pair_mul_prev");
        s->pair_mul_cur = mod_b("pair_mul_cur");
    }
    s->token_shift = geti(s, "token_shift", 0);
    const std::string block = gets(s, "block", "parallel"), residual = gets(s, "residual", "gated");
    s->sequential = block == "sequential";
    s->hyper = residual == "hyper";
    s->plain = residual == "plain";
    s->side_by_side = s->plain && !s->sequential;
    s->post_norm = geti(s, "post_norm", 0);
    s->resid_mult = (float) getd(s, "residual_mult", 1.0);
    s->tied_head = geti(s, "tied_head", 0);
    s->embed_norm = geti(s, "embedding_norm", 0);
    s->loop_input = geti(s, "loop_input", 1);
    s->side_dim = geti(s, "token_side", 0);
    s->logit_scale = (float) getd(s, "logit_scale", 1.0);
    s->logit_cap = (float) getd(s, "logit_softcap", 0.0);
    const int L = geti(s, "num_layers", 0);
    auto fail = [&](const char* why) {
        set_error("tllm_stack_create: %s", why);
        delete s;
        return (tllm_stack_t) nullptr;
    };
    if (s->width < 1 || s->vocab < 1 || L < 1)
        return fail("width, vocab and num_layers must be positive");
    if (s->groups < 1 || s->width % s->groups)
        return fail("width must split into norm_groups equal parts");
    if (s->page < 1 || s->blocks < 1 || s->slots < 1)
        return fail("page_size, num_blocks and num_slots must be positive");
    if ((block != "parallel" && block != "sequential") || (residual != "gated" && residual != "hyper" && residual != "plain") || (s->sequential ? residual == "gated" : s->hyper))
        return fail("block=parallel goes with residual=gated or plain, block=sequential with residual=hyper or plain");
    if ((s->embed_norm && !s->plain) || (s->side_dim && !s->side_by_side))
        return fail("the embedding norm is built for residual=plain, the per-layer token input for block=parallel, residual=plain");
    if ((s->post_norm || s->resid_mult != 1.f) && !(s->sequential && s->plain))
        return fail("post_norm and residual_mult are built for block=sequential, residual=plain");
    if (s->plain && (s->groups != 1 || s->loop_input))
        return fail("residual=plain goes with norm_groups=1 and loop_input=0");
    if (!s->plain && !s->loop_input)
        return fail("loop_input=0 is built for residual=plain");
    if (s->side_dim < 0 || s->logit_cap < 0)
        return fail("token_side and logit_softcap must not be negative");
    if (s->streams < 1 || s->streams > 8 || (!s->hyper && s->streams != 1))
        return fail("streams: 1 to 8, more than one only with residual=hyper");
    if (s->hyper && s->loop_stop > s->loop_start)
        return fail("looped layers are built for the gated residual only");
    if (s->pair_buckets < 0 || (s->token_shift && !s->hyper) || (s->pair_buckets && s->plain))
        return fail("pair_buckets >= 0, not with residual=plain; the token shift is built for block=sequential");
    s->last_tok.assign((size_t) s->slots, -1);
    s->fed.assign((size_t) s->slots, 0);
    if (s->loop_times < 1 || s->loop_start < 0 || s->loop_stop < s->loop_start || s->loop_stop > L)
        return fail("the loop must satisfy 0 <= loop_start <= loop_stop <= num_layers, loop_times >= 1");
    s->layers.resize(L);
    for (int i = 0; i < L; ++i)
    {
        Layer& l = s->layers[i];
        const std::string p = "layer." + std::to_string(i) + ".";
        const std::string kind = gets(s, p + "type", "");
        if (kind == "attention")
            l.kind = MIX_ATTENTION;
        else if (kind == "hgrn2")
            l.kind = MIX_HGRN2;
        else if (kind == "latent_attention")
            l.kind = MIX_LATENT;
        else if (kind == "mamba2")
            l.kind = MIX_MAMBA2;
        else if (kind == "delta_rule")
            l.kind = MIX_DELTA;
        else
        {
            set_error("tllm_stack_create: layer %d has mixer type '%s' (attention | latent_attention | hgrn2 | mamba2 | delta_rule)", i, kind.c_str());
            delete s;
            return nullptr;
        }
        l.heads = geti(s, p + "heads", 0);
        l.dim = geti(s, p + (l.kind == MIX_MAMBA2 ? "state" : "dim"), 0);
        l.vdim = geti(s, p + "vdim", l.dim);
        l.weights_of = geti(s, p + "weights_of", -1);
        if (l.weights_of >= i || (l.weights_of >= 0 && s->layers[l.weights_of].weights_of >= 0))
            return fail("weights_of names an earlier layer that has weights of its own");
        l.ff = geti(s, p + "ff", 0);
        if (l.heads < 1 || l.dim < 1 || l.vdim < 1 || l.ff < 0)
            return fail("a layer needs heads, dim and vdim");
        l.n_ctx = l.heads * l.vdim;
        const std::string mlp = gets(s, p + "mlp", "gelu_gate");
        if (mlp != "gelu_gate" && mlp != "relu2" && mlp != "moe")
            return fail("a layer's mlp is gelu_gate, relu2 or moe");
        l.mlp = mlp == "relu2" ? MLP_RELU2 : (mlp == "moe" ? MLP_MOE : MLP_GELU_GATE);
        if (l.mlp != MLP_GELU_GATE && !s->sequential && !s->plain)
            return fail("the relu2 and moe feed-forwards are built for block=sequential and for residual=plain");
        if (s->side_by_side && l.ff > 0 && l.mlp != MLP_MOE)
            return fail("block=parallel, residual=plain is built for the moe feed-forward");
        if ((l.kind == MIX_MAMBA2 || l.kind == MIX_DELTA || l.weights_of >= 0) && !s->sequential)
            return fail("mamba2 and delta_rule layers and shared weights are built for block=sequential");
        if (l.mlp == MLP_MOE && l.ff > 0)
        {
            l.experts = geti(s, p + "experts", 0);
            l.identity = geti(s, p + "identity", 0);
            l.top = geti(s, p + "top", 1);
            l.route_groups = geti(s, p + "route_groups", 1);
            l.route_keep = geti(s, p + "route_keep", l.route_groups);
            l.route_scale = getd(s, p + "route_scale", 1.0);
            const std::string rs = gets(s, p + "route_score", "softmax"), rw = gets(s, p + "route_weight", "output");
            if ((rs != "softmax" && rs != "sigmoid") || (rw != "output" && rw != "input"))
                return fail("moe: route_score softmax | sigmoid, route_weight output | input");
            const std::string ex = gets(s, p + "expert", "silu_gate");
            if (ex != "silu_gate" && ex != "relu2")
                return fail("moe: expert silu_gate | relu2");
            l.expert_relu2 = ex == "relu2";
            l.route_norm = geti(s, p + "route_norm", 0);
            l.shared_ff = geti(s, p + "shared_ff", 0);
            l.route_bias = geti(s, p + "route_bias", 0);
            l.shared_gate = geti(s, p + "shared_gate", 0);
            if (l.shared_ff < 0 || (l.shared_gate && l.shared_ff == 0) || (s->side_by_side && l.shared_ff > 0 && (!l.expert_relu2 || l.shared_gate)))
                return fail("moe: shared_gate goes with shared_ff; under block=parallel the shared expert is built for the relu2 form without a gate");
            l.n_shared = l.expert_relu2 ? l.shared_ff : 2 * l.shared_ff;
            l.route_sigmoid = rs == "sigmoid";
            l.route_weight_input = rw == "input";
            const int ne = l.experts + l.identity;
            if (l.experts < 1 || l.identity < 0 || ne > 1024 || l.top < 1 || l.top > 64 || l.top > ne || l.route_groups < 1 || ne % l.route_groups
                || l.route_keep < 1 || l.route_keep > l.route_groups)
                return fail("moe: experts >= 1, experts + identity <= 1024 in equal route_groups, 1 <= route_keep <= route_groups, top <= 64");
            s->max_top = std::max(s->max_top, l.top);
            s->max_experts = std::max(s->max_experts, l.experts);
            s->max_outputs = std::max(s->max_outputs, ne);
        }
        l.n_rg = (s->hyper || s->plain) ? 0 : s->width;
        if (s->side_by_side && l.kind != MIX_ATTENTION && l.kind != MIX_LATENT)
            return fail("block=parallel, residual=plain is built for attention and latent_attention layers");
        if (l.kind == MIX_LATENT)
        {
            l.kv_rank = geti(s, p + "kv_rank", 0);
            l.rot_part = geti(s, p + "rot_dim", 0);
            l.rot_dims = geti(s, p + "rot_dims", l.rot_part);
            l.rot_base = getd(s, p + "rot_base", 10000);
            l.rot_factor = getd(s, p + "rot_factor", 0);
            l.rot_original = getd(s, p + "rot_original", 0);
            l.rot_fast = getd(s, p + "rot_fast", 0);
            l.rot_slow = getd(s, p + "rot_slow", 0);
            l.scale = getd(s, p + "scale", 1.0 / std::sqrt((double) (l.dim + l.rot_part)));
            l.q_rank = geti(s, p + "q_rank", 0);
            const std::string pairing = gets(s, p + "rot_pairing", "neighbours"), mk = gets(s, p + "mask", "causal");
            if ((pairing != "neighbours" && pairing != "halves") || (mk != "causal" && mk != "window" && mk != "chunk"))
                return fail("latent_attention: rot_pairing neighbours | halves, mask causal | window | chunk");
            l.rot_halves = pairing == "halves";
            l.mask = mk == "window" ? MASK_WINDOW : (mk == "chunk" ? MASK_CHUNK : MASK_CAUSAL);
            l.mask_size = geti(s, p + "mask_size", 0);
            l.sink = geti(s, p + "sink", 0);
            l.out_gate = geti(s, p + "out_gate", 0);
            l.n_gate = l.out_gate ? l.heads : 0;
            if (l.kv_rank < 1 || l.rot_part < 0 || l.rot_dims < 0 || (l.rot_dims & 1) || l.rot_dims > l.rot_part || l.q_rank < 0)
                return fail("latent_attention: kv_rank positive, rot_dims even and <= rot_dim");
            if (l.mask != MASK_CAUSAL && l.mask_size < 1)
                return fail("latent_attention: a window or chunk mask needs mask_size >= 1");
            l.kv_heads = 1;
            // columns of the mixer's projection: the queries of every head, or the query latent they are expanded from
            l.n_q = l.q_rank > 0 ? l.q_rank : l.heads * (l.dim + l.rot_part);
            l.n_k = l.kv_rank + l.rot_part; // the down projection: latent | rotated key part
            l.n_v = 0;
            s->max_qrank = std::max(s->max_qrank, l.q_rank);
            if (l.q_rank > 0)
                s->max_qfull = std::max(s->max_qfull, l.heads * (l.dim + l.rot_part));
            l.n_lat = l.heads * l.kv_rank;
            s->max_lat = std::max(s->max_lat, l.n_lat);
            s->max_q = std::max(s->max_q, l.heads * (l.kv_rank + l.rot_part));
        }
        else if (l.kind == MIX_ATTENTION)
        {
            l.qkv_bias = geti(s, p + "qkv_bias", 0);
            l.qk_norm = geti(s, p + "qk_norm", 0);
            l.head_temp = geti(s, p + "head_temp", 0);
            const std::string pb = gets(s, p + "pos_bias", "none"), mk = gets(s, p + "mask", "causal"), wt = gets(s, p + "weights", "softmax");
            if ((pb != "none" && pb != "linear" && pb != "log") || (mk != "causal" && mk != "window" && mk != "chunk")
                || (wt != "softmax" && wt != "sigmoid"))
                return fail("attention: pos_bias none | linear | log, mask causal | window | chunk, weights softmax | sigmoid");
            l.pos_bias = pb == "linear" ? 1 : (pb == "log" ? 2 : 0);
            l.slope_base = getd(s, p + "slope_base", 8.0);
            l.mask = mk == "window" ? MASK_WINDOW : (mk == "chunk" ? MASK_CHUNK : MASK_CAUSAL);
            l.mask_size = geti(s, p + "mask_size", 0);
            l.weights = wt == "sigmoid" ? WEIGHTS_SIGMOID : WEIGHTS_SOFTMAX;
            l.sink = geti(s, p + "sink", 0);
            l.out_gate = geti(s, p + "out_gate", 0);
            l.mask_keep = geti(s, p + "mask_keep", 0);
            l.talk = geti(s, p + "talk", 0);
            l.values_are_keys = geti(s, p + "values_are_keys", 0);
            l.gate_wide = geti(s, p + "gate_wide", 0);
            l.qk_norm_weight = geti(s, p + "qk_norm_weight", 0);
            l.o_bias = geti(s, p + "o_bias", 0);
            const std::string rsc = gets(s, p + "rot_scaling", "yarn");
            const std::string pairing = gets(s, p + "rot_pairing", "neighbours");
            if ((rsc != "yarn" && rsc != "banded" && rsc != "linear") || (pairing != "neighbours" && pairing != "halves"))
                return fail("attention: rot_scaling yarn | banded | linear, rot_pairing neighbours | halves");
            l.rot_banded = rsc == "banded";
            l.rot_linear = rsc == "linear";
            l.rot_halves = pairing == "halves";
            l.v_mix = geti(s, p + "v_mix", 0);
            l.rot_low = getd(s, p + "rot_low", 1.0);
            l.rot_high = getd(s, p + "rot_high", 4.0);
            if (l.rot_banded && !(l.rot_high > l.rot_low && l.rot_low > 0))
                return fail("attention: banded frequency scaling needs 0 < rot_low < rot_high");
            if (l.mask != MASK_CAUSAL && l.mask_size < 1)
                return fail("attention: a window or chunk mask needs mask_size >= 1");
            if (l.mask_keep < 0 || (l.mask_keep > 0 && l.mask != MASK_WINDOW) || (l.values_are_keys && l.vdim != l.dim)
                || (l.gate_wide && !l.out_gate) || (l.qk_norm_weight && !l.qk_norm) || (l.o_bias && !s->sequential))
                return fail("attention: mask_keep goes with a window, values_are_keys with vdim = dim, gate_wide with out_gate, qk_norm_weight "
                            "with qk_norm, o_bias with block=sequential");
            if (l.sink && l.weights == WEIGHTS_SIGMOID)
                return fail("attention: a sink belongs to softmax weights");
            l.n_gate = l.out_gate ? (l.gate_wide ? l.heads * l.vdim : l.heads) : 0;
            l.kv_heads = geti(s, p + "kv_heads", l.heads);
            l.maps = geti(s, p + "maps", 1);
            l.diff = getd(s, p + "diff", 0);
            l.scale = getd(s, p + "scale", 1.0 / std::sqrt((double) l.dim));
            l.softcap = getd(s, p + "softcap", 0);
            l.head_norm = geti(s, p + "head_norm", 0);
            l.rot_dims = geti(s, p + "rot_dims", 0);
            l.rot_base = getd(s, p + "rot_base", 10000);
            l.rot_factor = getd(s, p + "rot_factor", 0);
            l.rot_original = getd(s, p + "rot_original", 0);
            l.rot_fast = getd(s, p + "rot_fast", 0);
            l.rot_slow = getd(s, p + "rot_slow", 0);
            if (l.kv_heads < 1 || l.heads % l.kv_heads || l.maps < 1 || l.maps > 2 || (l.rot_dims > 0 && (l.dim & 1) && !l.rot_halves) || (l.rot_dims & 1)
                || l.rot_dims > l.dim)
                return fail("attention: heads must be a multiple of kv_heads, maps 1 or 2, rot_dims even and <= dim, dim even where neighbours turn");
            if (l.talk && (l.maps != 1 || l.weights != WEIGHTS_SOFTMAX || l.softcap > 0 || l.head_norm || l.head_temp || l.pos_bias))
                return fail("attention: talking heads go with one plain softmax map");
            if (l.talk)
                s->max_pairs = std::max(s->max_pairs, l.heads * l.kv_heads * l.vdim);
            l.n_q = l.heads * l.maps * l.dim;
            l.n_k = l.kv_heads * l.maps * l.dim;
            l.n_v = l.values_are_keys ? 0 : l.kv_heads * l.vdim; // columns of the projection; the cache holds value rows either way
            if (l.v_mix)
            {
                if (s->v_mix_first < 0)
                    s->v_mix_first = i, s->v_mix_cols = l.kv_heads * l.vdim;
                if (l.kv_heads * l.vdim != s->v_mix_cols || l.weights_of >= 0 || s->loop_stop > s->loop_start)
                    return fail("attention: layers that mix values have equally many values per token and weights of their own; no loop");
            }
        }
        else if (l.kind == MIX_MAMBA2)
        {
            l.groups = geti(s, p + "groups", 1);
            l.taps = geti(s, p + "conv", 4);
            l.ssm_norm_groups = geti(s, p + "ssm_norm_groups", 1);
            if (l.groups < 1 || l.heads % l.groups || l.ssm_norm_groups < 1 || (l.heads * l.vdim) % l.ssm_norm_groups
                || !stack_ssm_serves(l.vdim, l.dim, l.taps))
                return fail("mamba2: heads a multiple of groups, heads * vdim a multiple of ssm_norm_groups, conv 1 .. 16, state x vdim up to 32 x 1024");
            // columns of the projection: z | x | B | C | dt; the convolution runs over x | B | C
            l.n_conv = l.heads * l.vdim + 2 * l.groups * l.dim;
            l.n_q = l.heads * l.vdim;
            l.n_k = l.n_conv;
            l.n_v = l.heads;
            s->max_conv = std::max(s->max_conv, l.n_conv);
        }
        else if (l.kind == MIX_DELTA)
        {
            l.kv_heads = geti(s, p + "kv_heads", l.heads);
            l.taps = geti(s, p + "conv", 4);
            l.decay_rank = geti(s, p + "decay_rank", 0);
            l.gate_rank = geti(s, p + "gate_rank", 0);
            if (l.kv_heads < 1 || l.heads % l.kv_heads || l.taps < 1 || l.taps > 16 || l.decay_rank < 1 || l.gate_rank < 1
                || !stack_delta_serves(l.dim, l.vdim))
                return fail("delta_rule: heads a multiple of kv_heads, conv 1 .. 16, decay_rank and gate_rank positive, dim up to 512");
            // columns of the projection: q | k | v (the convolution's channels) | beta, padded to 8 | decay latent | gate latent
            l.n_q = l.kv_heads * l.dim;
            l.n_k = l.kv_heads * l.dim;
            l.n_v = l.heads * l.vdim;
            l.n_conv = l.n_q + l.n_k + l.n_v;
            l.n_beta = (l.heads + 7) / 8 * 8;
            l.n_gate = l.n_beta + l.decay_rank + l.gate_rank;
            l.n_gate = (l.n_conv + l.n_gate + 7) / 8 * 8 - l.n_conv; // rows of the element type stay 16-byte aligned
            s->max_conv = std::max(s->max_conv, l.n_conv);
            s->max_hd = std::max(s->max_hd, l.heads * l.dim);
        }
        else
        {
            if (!stack_hgrn2_serves(l.dim, l.vdim))
                return fail("hgrn2: dim up to 512");
            l.n_q = l.heads * l.dim;
            l.n_k = l.heads * l.dim; // forget gate
            l.n_v = l.heads * l.vdim;
        }
        l.n_mix = l.n_q + l.n_k + l.n_v + l.n_rg + l.n_gate;
        if (s->side_by_side)
        {
            // zero rows up to a multiple of 8 (rows of the element type stay 16-byte aligned); the router's columns follow the shared expert's
            l.n_pad = (l.n_mix + 7) / 8 * 8 - l.n_mix;
            l.n_mix += l.n_pad;
            l.n_route = l.mlp == MLP_MOE && l.ff > 0 ? l.experts + l.identity : 0;
        }
        s->max_sh = std::max(s->max_sh, l.shared_ff);
        const int ff_rows = l.mlp == MLP_MOE ? l.top : 1; // a mixture's products run on one row per (token, chosen expert)
        s->max_proj = std::max(s->max_proj, std::max(l.n_mix, l.n_rg));
        s->max_q = std::max(s->max_q, l.n_q);
        s->max_ctx = std::max(s->max_ctx, l.n_ctx + (s->side_by_side ? l.shared_ff : 0));
        s->max_ff = std::max(s->max_ff, ff_rows * l.ff);
    }
    // execution order
    auto add = [&](int layer, int pass, bool enters) {
        Run r;
        r.layer = layer;
        r.pass = pass;
        r.enters_pass = enters;
        s->runs.push_back(r);
    };
    const bool looped = s->loop_stop > s->loop_start;
    for (int i = 0; i < (looped ? s->loop_start : L); ++i)
        add(i, 0, false);
    if (looped)
    {
        for (int t = 0; t < s->loop_times; ++t)
            for (int i = s->loop_start; i < s->loop_stop; ++i)
                add(i, t, i == s->loop_start);
        for (int i = s->loop_stop; i < L; ++i)
            add(i, 0, false);
    }
    return s;
}

int32_t tllm_stack_set_tensor(tllm_stack_t s, const char* name, int32_t dtype, const int64_t* dims, int32_t nbDims, const void* data)
{
    if (!s || !name || !data || nbDims < 0 || nbDims > 4 || s->finalized)
    {
        set_error("tllm_stack_set_tensor: bad arguments (or the engine is already finalized)");
        return -1;
    }
    HostTensor t;
    for (int i = 0; i < nbDims; ++i)
        t.dims.push_back(dims[i]);
    const int64_t n = t.numel();
    t.v.resize((size_t) n);
    if (dtype == DT_FLOAT)
        std::memcpy(t.v.data(), data, (size_t) n * 4);
    else if (dtype == DT_BF16)
    {
        const uint16_t* b = static_cast<const uint16_t*>(data);
        for (int64_t i = 0; i < n; ++i)
        {
            const uint32_t u = (uint32_t) b[i] << 16;
            std::memcpy(&t.v[(size_t) i], &u, 4);
        }
    }
    else
    {
        set_error("tllm_stack_set_tensor(%s): dtype %d (0 = fp32, 7 = bfloat16)", name, dtype);
        return -1;
    }
    s->host[name] = std::move(t);
    return 0;
}

int32_t tllm_stack_finalize(tllm_stack_t s)
{
    if (!s || s->finalized)
    {
        set_error("tllm_stack_finalize: no engine, or finalized twice");
        return -1;
    }
    const int64_t Wd = s->width;
    const HostTensor* t = need(s, "embed", {s->vocab, Wd});
    if (!t || upload_rows(s, {t}, &s->embed))
        return -1;
    if (s->tied_head)
        s->head = s->embed;
    else
    {
        t = need(s, "head", {s->vocab, Wd});
        if (!t || upload_rows(s, {t}, &s->head))
            return -1;
    }
    // a norm weight as the kernels apply it: the stored value plus the design's offset (0, or 1 for weights stored around zero)
    auto norm_vec = [&](const std::string& name, int64_t len, float** out) {
        const HostTensor* v = need(s, name, {len});
        if (!v)
            return -1;
        std::vector<float> w(v->v);
        for (float& f : w)
            f += s->norm_offset;
        return upload_f32(s, w.data(), w.size(), out);
    };
    auto norm_plain = [&](const std::string& name, int64_t len, float** out) {
        const HostTensor* v = need(s, name, {len});
        return (!v || upload_f32(s, v->v.data(), v->v.size(), out)) ? -1 : 0;
    };
    if (norm_vec("final.norm", Wd, &s->final_norm))
        return -1;
    {
        const std::vector<float> one(64, 1.f);
        if (upload_f32(s, one.data(), one.size(), &s->ones))
            return -1;
    }
    if (s->embed_norm && norm_vec("embed.norm", Wd, &s->embed_norm_w))
        return -1;
    if (s->side_dim > 0)
    {
        t = need(s, "side.embed", {s->vocab, (int64_t) s->side_dim * (int64_t) s->layers.size()});
        if (!t || upload_rows(s, {t}, &s->side_embed))
            return -1;
    }
    if (s->pair_buckets > 0)
    {
        t = need(s, "bigram", {s->pair_buckets + 1, Wd});
        if (!t || upload_rows(s, {t}, &s->pair_table))
            return -1;
    }
    if (s->loop_stop > s->loop_start)
    {
        t = need(s, "loop.step", {s->loop_times, Wd});
        if (!t || upload_f32(s, t->v.data(), t->v.size(), &s->loop_step))
            return -1;
    }
    for (size_t i = 0; i < s->layers.size(); ++i)
    {
        Layer& l = s->layers[i];
        const std::string p = "l" + std::to_string(i) + ".";
        auto vec = [&](const std::string& n, int64_t len, float** out) {
            const HostTensor* v = need(s, p + n, {len});
            return (!v || upload_f32(s, v->v.data(), v->v.size(), out)) ? -1 : 0;
        };
        if (l.weights_of >= 0)
        {
            // the layer runs on another layer's weights: same description, same device tensors; caches and states go by run
            const Layer& src = s->layers[(size_t) l.weights_of];
            if (src.kind != l.kind || src.n_mix != l.n_mix || src.n_ctx != l.n_ctx || src.ff != l.ff || src.mlp != l.mlp || src.dim != l.dim
                || src.heads != l.heads || src.shared_ff != l.shared_ff || src.experts != l.experts || src.identity != l.identity || src.kv_rank != l.kv_rank
                || src.rot_part != l.rot_part || src.taps != l.taps)
            {
                set_error("tllm_stack_finalize: layer %d uses the weights of layer %d, but their shapes differ", (int) i, l.weights_of);
                return -1;
            }
            const int from = l.weights_of;
            l = src;
            l.weights_of = from;
            continue;
        }
        if (norm_vec(p + "norm1", Wd, &l.norm1) || (s->post_norm && norm_vec(p + "norm1b", Wd, &l.norm1b))
            || (s->post_norm && l.ff > 0 && norm_vec(p + "norm2b", Wd, &l.norm2b)))
            return -1;
        if (s->token_shift && vec("shift", Wd, &l.shift))
            return -1;
        if (s->side_dim > 0)
        {
            const HostTensor *sg = need(s, p + "side.gate", {s->side_dim, Wd}), *sp = need(s, p + "side.proj", {Wd, s->side_dim});
            if (!sg || !sp || upload_rows(s, {sg}, &l.side_gate) || upload_rows(s, {sp}, &l.side_proj) || norm_plain(p + "side.norm", Wd, &l.side_norm))
                return -1;
        }
        const HostTensor* rg1 = nullptr;
        if (s->plain)
            ; // neither gates nor connections
        else if (!s->hyper)
        {
            rg1 = need(s, p + "rg1", {Wd, Wd});
            if (!rg1 || vec("rg1.b", Wd, &l.rg1_b))
                return -1;
        }
        else
        {
            // hyper-connections of the two sublayers; a model with one plain stream has no such tensors: mix = out = in = 1
            for (int q = 0; q < 2; ++q)
            {
                HyperW& hw = l.hc[q];
                const std::string hp = "hc" + std::to_string(q + 1) + ".";
                if (s->host.count(p + hp + "mix") == 0 && s->streams == 1)
                {
                    hw.mix = hw.out = hw.in = s->ones;
                    continue;
                }
                if (q == 1 && l.ff == 0)
                    continue;
                const HostTensor* m = need(s, p + hp + "mix", {s->streams, s->streams});
                if (!m || upload_f32(s, m->v.data(), m->v.size(), &hw.mix) || vec(hp + "out", s->streams, &hw.out)
                    || vec(hp + "in", s->streams, &hw.in))
                    return -1;
            }
        }
        if (l.kind == MIX_MAMBA2)
        {
            const HostTensor* win = need(s, p + "mix.in", {l.n_mix, Wd});
            const HostTensor* wo = need(s, p + "mix.o", {Wd, l.n_ctx});
            const HostTensor* cw = need(s, p + "mix.conv", {l.n_conv, l.taps});
            if (!win || !wo || !cw || upload_rows(s, {win}, &l.w_mix) || upload_rows(s, {wo}, &l.w_o)
                || upload_f32(s, cw->v.data(), cw->v.size(), &l.conv_w) || vec("mix.conv.b", l.n_conv, &l.conv_b)
                || vec("mix.dt_bias", l.heads, &l.dt_bias) || vec("mix.A_log", l.heads, &l.a_log) || vec("mix.D", l.heads, &l.d_skip)
                || vec("mix.norm", l.n_ctx, &l.hnorm))
                return -1;
        }
        if (l.kind == MIX_DELTA)
        {
            const int64_t QK = l.n_q, HV = l.n_v, HD = (int64_t) l.heads * l.dim;
            const HostTensor *wq = need(s, p + "mix.q", {QK, Wd}), *wk = need(s, p + "mix.k", {QK, Wd}), *wv = need(s, p + "mix.v", {HV, Wd}),
                             *wb = need(s, p + "mix.b", {l.heads, Wd}), *a1 = need(s, p + "mix.a1", {l.decay_rank, Wd}),
                             *a2 = need(s, p + "mix.a2", {HD, l.decay_rank}), *g1 = need(s, p + "mix.g1", {l.gate_rank, Wd}),
                             *g2 = need(s, p + "mix.g2", {HV, l.gate_rank}), *wo = need(s, p + "mix.o", {Wd, HV}),
                             *cq = need(s, p + "mix.q.conv", {QK, l.taps}), *ck = need(s, p + "mix.k.conv", {QK, l.taps}),
                             *cv = need(s, p + "mix.v.conv", {HV, l.taps});
            if (!wq || !wk || !wv || !wb || !a1 || !a2 || !g1 || !g2 || !wo || !cq || !ck || !cv)
                return -1;
            l.low_pair = HD == HV && l.decay_rank == l.gate_rank;
            HostTensor pad_b, pad_end; // zero rows: beta's columns up to a multiple of 8, the projection's up to a multiple of 8
            pad_b.dims = {l.n_beta - l.heads, Wd};
            pad_b.v.assign((size_t) pad_b.numel(), 0.f);
            pad_end.dims = {l.n_gate - l.n_beta - l.decay_rank - l.gate_rank, Wd};
            pad_end.v.assign((size_t) pad_end.numel(), 0.f);
            std::vector<float> taps(cq->v);
            taps.insert(taps.end(), ck->v.begin(), ck->v.end());
            taps.insert(taps.end(), cv->v.begin(), cv->v.end());
            if (upload_rows(s, {wq, wk, wv, wb, &pad_b, a1, g1, &pad_end}, &l.w_mix) || upload_rows(s, {wo}, &l.w_o)
                || (l.low_pair ? upload_rows(s, {a2, g2}, &l.w_a2) : upload_rows(s, {a2}, &l.w_a2) || upload_rows(s, {g2}, &l.w_g2)) || upload_f32(s, taps.data(), taps.size(), &l.conv_w) || vec("mix.dt_bias", HD, &l.dt_bias)
                || vec("mix.A_log", l.heads, &l.a_log) || vec("mix.norm", l.vdim, &l.hnorm))
                return -1;
        }
        const bool own_mix = l.kind == MIX_MAMBA2 || l.kind == MIX_DELTA; // kinds whose projection is put together above
        const bool q_latent = l.kind == MIX_LATENT && l.q_rank > 0;
        const HostTensor* wq = own_mix ? nullptr : need(s, p + (q_latent ? "mix.dq" : "mix.q"), {l.n_q, Wd});
        const HostTensor* wk = own_mix
            ? nullptr
            : need(s, p + (l.kind == MIX_ATTENTION ? "mix.k" : (l.kind == MIX_LATENT ? "mix.dkv" : "mix.f")), {l.n_k, Wd});
        const HostTensor* wv = (l.kind == MIX_LATENT || own_mix || l.values_are_keys) ? nullptr : need(s, p + "mix.v", {l.n_v, Wd});
        const HostTensor* wo = own_mix ? nullptr : need(s, p + "mix.o", {Wd, l.n_ctx});
        const HostTensor* wg = l.n_gate ? need(s, p + "mix.g", {l.n_gate, Wd}) : nullptr;
        if (!own_mix && (!wq || !wk || (!wv && l.kind != MIX_LATENT && !l.values_are_keys) || !wo || (l.n_gate && !wg)))
            return -1;
        if (!own_mix)
        {
            std::vector<const HostTensor*> rows = {wq, wk};
            if (wv)
                rows.push_back(wv);
            if (rg1)
                rows.push_back(rg1);
            if (wg)
                rows.push_back(wg);
            HostTensor pad, joint;
            const HostTensor* out_w = wo;
            if (s->side_by_side)
            {
                // everything else that reads the layer's one normed row: the shared expert's up rows and the router's
                pad.dims = {l.n_pad, Wd};
                pad.v.assign((size_t) pad.numel(), 0.f);
                rows.push_back(&pad);
                if (l.shared_ff > 0)
                {
                    const HostTensor *su = need(s, p + "mlp.shared.up", {l.shared_ff, Wd}), *sd = need(s, p + "mlp.shared.down", {Wd, l.shared_ff});
                    if (!su || !sd)
                        return -1;
                    rows.push_back(su);
                    if (l.kind == MIX_LATENT)
                    {
                        // [Wo | Wshared_down]: context and shared activations lie side by side in one row
                        const int64_t A = l.n_ctx, B = l.shared_ff;
                        joint.dims = {Wd, A + B};
                        joint.v.resize((size_t) (Wd * (A + B)));
                        for (int64_t n = 0; n < Wd; ++n)
                        {
                            std::copy_n(wo->v.data() + n * A, A, joint.v.data() + n * (A + B));
                            std::copy_n(sd->v.data() + n * B, B, joint.v.data() + n * (A + B) + A);
                        }
                        out_w = &joint;
                    }
                    else if (upload_rows(s, {sd}, &l.w_shared_down))
                        return -1;
                }
                if (l.n_route > 0)
                {
                    const HostTensor* rw = need(s, p + "mlp.router", {l.n_route, Wd});
                    if (!rw)
                        return -1;
                    rows.push_back(rw);
                }
            }
            if (upload_rows(s, rows, &l.w_mix) || upload_rows(s, {out_w}, &l.w_o))
                return -1;
        }
        if (l.kind == MIX_ATTENTION || l.kind == MIX_LATENT)
        {
            std::vector<float> fr((size_t) std::max(l.rot_dims / 2, 1));
            if (l.rot_linear)
                stack_rope_freqs_linear(fr.data(), l.rot_dims, l.rot_base, l.rot_factor), l.mscale = 1.f;
            else if (l.rot_banded)
                stack_rope_freqs_banded(fr.data(), l.rot_dims, l.rot_base, l.rot_factor, l.rot_original, l.rot_low, l.rot_high), l.mscale = 1.f;
            else
                l.mscale = stack_rope_freqs(fr.data(), l.rot_dims, l.rot_base, l.rot_factor, l.rot_original, l.rot_fast, l.rot_slow);
            if (upload_f32(s, fr.data(), fr.size(), &l.freq))
                return -1;
        }
        if (l.kind == MIX_LATENT)
        {
            const int64_t C = l.kv_rank, D = l.dim, E = l.vdim, H = l.heads;
            const HostTensor* uk = need(s, p + "mix.uk", {H * D, C});
            const HostTensor* uv = need(s, p + "mix.uv", {H * E, C});
            if (!uk || !uv || norm_plain(p + "mix.dkv.norm", C, &l.lat_norm))
                return -1;
            if (q_latent)
            {
                const HostTensor* uq = need(s, p + "mix.uq", {H * (D + l.rot_part), l.q_rank});
                if (!uq || upload_rows(s, {uq}, &l.w_uq) || norm_plain(p + "mix.dq.norm", l.q_rank, &l.cq_norm))
                    return -1;
            }
            if (l.sink && vec("mix.sink", l.heads, &l.sinkv))
                return -1;
            // W_uk^T per head, [kv_rank, dim]: the query side of the absorbed score is a product with these rows
            HostTensor tr;
            tr.dims = {H * C, D};
            tr.v.resize((size_t) (H * C * D));
            for (int64_t h = 0; h < H; ++h)
                for (int64_t d = 0; d < D; ++d)
                    for (int64_t c = 0; c < C; ++c)
                        tr.v[(size_t) ((h * C + c) * D + d)] = uk->v[(size_t) ((h * D + d) * C + c)];
            if (upload_rows(s, {&tr}, &l.w_ukT) || upload_rows(s, {uv}, &l.w_uv))
                return -1;
        }
        else if (l.kind == MIX_ATTENTION)
        {
            l.lambda = 0.f;
            if (l.maps == 2)
            {
                const HostTensor *a1 = need(s, p + "mix.lq1", {l.dim}), *b1 = need(s, p + "mix.lk1", {l.dim}),
                                 *a2 = need(s, p + "mix.lq2", {l.dim}), *b2 = need(s, p + "mix.lk2", {l.dim});
                if (!a1 || !b1 || !a2 || !b2)
                    return -1;
                float d1 = 0.f, d2 = 0.f;
                for (int d = 0; d < l.dim; ++d)
                {
                    d1 += a1->v[d] * b1->v[d];
                    d2 += a2->v[d] * b2->v[d];
                }
                l.lambda = std::exp(d1) - std::exp(d2) + (float) l.diff;
            }
            if (l.qkv_bias)
            {
                const HostTensor *bq = need(s, p + "mix.q.b", {l.n_q}), *bk = need(s, p + "mix.k.b", {l.n_k}),
                                 *bv = l.values_are_keys ? nullptr : need(s, p + "mix.v.b", {l.n_v});
                if (!bq || !bk || (!bv && !l.values_are_keys))
                    return -1;
                std::vector<float> b(bq->v);
                b.insert(b.end(), bk->v.begin(), bk->v.end());
                if (bv)
                    b.insert(b.end(), bv->v.begin(), bv->v.end());
                b.resize((size_t) (l.n_mix + (s->side_by_side ? l.shared_ff + l.n_route : 0)), 0.f); // added by the product: nothing on its other columns
                if (upload_f32(s, b.data(), b.size(), &l.bias))
                    return -1;
            }
            if (l.v_mix && (int) i != s->v_mix_first)
            {
                const HostTensor* lam = s->host.count(p + "mix.vmix") ? &s->host[p + "mix.vmix"] : nullptr;
                if (!lam || lam->numel() != 1)
                {
                    set_error("tllm_stack_finalize: %smix.vmix is missing or not one number", p.c_str());
                    return -1;
                }
                l.vmix = lam->v[0];
            }
            if (l.head_temp && vec("mix.temp", l.heads, &l.temp))
                return -1;
            if (l.pos_bias == 1)
            {
                std::vector<float> sl((size_t) l.heads);
                for (int h = 0; h < l.heads; ++h)
                    sl[(size_t) h] = (float) std::exp2(-l.slope_base * (h + 1) / l.heads);
                if (upload_f32(s, sl.data(), sl.size(), &l.slope))
                    return -1;
            }
            if (l.pos_bias == 2 && (vec("mix.r1", l.heads, &l.r1) || vec("mix.r2", l.heads, &l.r2)))
                return -1;
            if (l.sink == 1 && vec("mix.sink", l.heads, &l.sinkv))
                return -1;
            if (l.sink == 2)
            {
                // a constant sink of logit 0: the softmax denominator holds one more 1
                const std::vector<float> zero((size_t) l.heads, 0.f);
                if (upload_f32(s, zero.data(), zero.size(), &l.sinkv))
                    return -1;
            }
            if (l.weights == WEIGHTS_SIGMOID && vec("mix.pb", l.heads, &l.wbias))
                return -1;
            if (l.talk)
            {
                const HostTensor* tk = need(s, p + "mix.talk", {l.heads, l.heads});
                if (!tk || upload_f32(s, tk->v.data(), tk->v.size(), &l.talkw))
                    return -1;
            }
            if (l.qk_norm_weight && (vec("mix.q.norm", l.dim, &l.q_norm) || vec("mix.k.norm", l.dim, &l.k_norm)))
                return -1;
            if (l.o_bias && vec("mix.o.b", Wd, &l.o_biasv))
                return -1;
        }
        else if (l.kind == MIX_HGRN2)
        {
            if (vec("mix.f.b", l.n_k, &l.f_bias) || vec("mix.lower", l.n_k, &l.lower) || vec("mix.norm", l.vdim, &l.hnorm))
                return -1;
        }
        if (l.ff > 0 && l.mlp == MLP_MOE)
        {
            // experts stacked: gate_e and up_e rows in turn per expert, then the down matrices; router and correction stay fp32
            const int ne = l.experts + l.identity;
            const HostTensor* rw = need(s, p + "mlp.router", {ne, Wd});
            if (!rw || (!s->side_by_side && norm_vec(p + "norm2", Wd, &l.norm2)) || (!s->plain && upload_f32(s, rw->v.data(), rw->v.size(), &l.router_w))
                || (l.route_bias && vec("mlp.router.b", ne, &l.route_b)))
                return -1;
            if (s->sequential)
            {
                // what reads the sublayer's row beside the experts: the shared expert's first matrices, the router (with residual=plain), the
                // shared expert's gate
                std::vector<const HostTensor*> first;
                if (l.shared_ff > 0)
                {
                    const HostTensor *su = l.expert_relu2 ? need(s, p + "mlp.shared.up", {l.shared_ff, Wd})
                                                          : need_gated(s, p + "mlp.shared.gate", p + "mlp.shared.up", l.shared_ff, Wd),
                                     *sd = need(s, p + "mlp.shared.down", {Wd, l.shared_ff});
                    if (!su || !sd || upload_rows(s, {sd}, &l.w_shared_down))
                        return -1;
                    first.push_back(su);
                }
                if (s->plain)
                    first.push_back(rw);
                if (l.shared_gate)
                {
                    const HostTensor* zg = need(s, p + "mlp.shared.sg", {1, Wd});
                    if (!zg)
                        return -1;
                    first.push_back(zg);
                }
                if (!first.empty() && upload_rows(s, first, &l.w_shared_up))
                    return -1;
            }
            if (s->host.count(p + "mlp.correction") && vec("mlp.correction", ne, &l.correction))
                return -1;
            std::vector<const HostTensor*> gu, dn;
            for (int e = 0; e < l.experts; ++e)
            {
                const std::string ep = p + "mlp.e" + std::to_string(e) + ".";
                const HostTensor *u = l.expert_relu2 ? need(s, ep + "up", {l.ff, Wd}) : need_gated(s, ep + "gate", ep + "up", l.ff, Wd),
                                 *d = need(s, ep + "down", {Wd, l.ff});
                if (!u || !d)
                    return -1;
                gu.push_back(u);
                dn.push_back(d);
            }
            if (upload_rows(s, gu, &l.w_gu) || upload_rows(s, dn, &l.w_down))
                return -1;
        }
        else if (l.ff > 0)
        {
            if (norm_vec(p + "norm2", Wd, &l.norm2))
                return -1;
            const HostTensor* rg2 = nullptr;
            if (!s->sequential)
            {
                rg2 = need(s, p + "rg2", {Wd, Wd});
                if (!rg2 || vec("rg2.b", Wd, &l.rg2_b))
                    return -1;
            }
            const HostTensor* wu = l.mlp == MLP_GELU_GATE ? need_gated(s, p + "mlp.gate", p + "mlp.up", l.ff, Wd) : need(s, p + "mlp.up", {l.ff, Wd});
            const HostTensor* wd = need(s, p + "mlp.down", {Wd, l.ff});
            if (!wu || !wd)
                return -1;
            std::vector<const HostTensor*> rows = {wu};
            if (rg2)
                rows.push_back(rg2);
            if (upload_rows(s, rows, &l.w_gu) || upload_rows(s, {wd}, &l.w_down))
                return -1;
        }
    }
    size_t ws_floats = 0;
    for (const Layer& l : s->layers)
        if (l.kind == MIX_ATTENTION)
            ws_floats = std::max(ws_floats, stack_attn_workspace_floats(l.talk ? l.heads * l.kv_heads : l.heads, l.maps, l.vdim));
        else if (l.kind == MIX_LATENT)
            ws_floats = std::max(ws_floats, stack_attn_workspace_floats(l.heads, 1, l.kv_rank));
    if (ws_floats)
    {
        void* ws = nullptr;
        if (alloc_zero(s, ws_floats * 4, &ws))
            return -1;
        s->attn_ws = (float*) ws;
    }
    for (Run& r : s->runs)
    {
        const Layer& l = s->layers[r.layer];
        if (l.kind == MIX_LATENT)
        {
            // one key row [latent | rotated part] and one value row (the latent, channel-major) per token, shared by all heads
            if (alloc_zero(s, (size_t) s->blocks * s->page * (l.kv_rank + l.rot_part) * s->es, &r.k_pool)
                || alloc_zero(s, (size_t) s->blocks * s->page * l.kv_rank * s->es, &r.v_pool))
                return -1;
        }
        else if (l.kind == MIX_ATTENTION)
        {
            if (alloc_zero(s, (size_t) s->blocks * l.kv_heads * l.maps * s->page * l.dim * s->es, &r.k_pool)
                || alloc_zero(s, (size_t) s->blocks * l.kv_heads * s->page * l.vdim * s->es, &r.v_pool))
                return -1;
        }
        else if (l.kind == MIX_MAMBA2 || l.kind == MIX_DELTA)
        {
            void *st = nullptr, *cv = nullptr;
            if (alloc_zero(s, (size_t) s->slots * l.heads * l.dim * l.vdim * 4, &st)
                || alloc_zero(s, (size_t) s->slots * l.taps * l.n_conv * 4, &cv))
                return -1;
            r.state = (float*) st;
            r.conv_state = (float*) cv;
        }
        else
        {
            void* st = nullptr;
            if (alloc_zero(s, (size_t) s->slots * l.heads * l.dim * l.vdim * 4, &st))
                return -1;
            r.state = (float*) st;
        }
        if (s->token_shift)
        {
            void* cr = nullptr;
            if (alloc_zero(s, (size_t) s->slots * s->width * 4, &cr))
                return -1;
            r.shift_carry = (float*) cr;
        }
    }
    s->host.clear();
    s->token_flops = 2.0 * (double) (tllm_stack_step_bytes(s, 1, 0, 0) / s->es - ((int64_t) s->vocab + 1) * s->width); // (of each weight that it meets)
    s->finalized = true;
    return 0;
}

int32_t tllm_stack_step(tllm_stack_t s, const tllm_stack_batch_t* b, float* logits_out, int32_t* next_ids_out, void* stream_v)
{
    if (!s || !s->finalized || !b)
    {
        set_error("tllm_stack_step: the engine is not finalized");
        return -1;
    }
    hipStream_t stream = (hipStream_t) stream_v;
    const int T = b->n_tokens, E = b->n_entries, NW = b->n_want, MB = b->max_blocks;
    if (T < 1 || E < 1 || NW < 0 || MB < 1 || !b->tokens || !b->ent_count || !b->ent_pos0 || !b->ent_slot || !b->block_table
        || (NW > 0 && !b->want_rows))
    {
        set_error("tllm_stack_step: empty batch or missing array");
        return -1;
    }
    // ---- every index the kernels will follow is checked here
    int64_t sum = 0;
    int max_count = 0, max_ctx = 0;
    for (int e = 0; e < E; ++e)
    {
        const int c = b->ent_count[e], p0 = b->ent_pos0[e], sl = b->ent_slot[e];
        if (c < 1 || p0 < 0 || sl < 0 || sl >= s->slots)
        {
            set_error("tllm_stack_step: entry %d has count %d, pos0 %d, slot %d (slots: %d)", e, c, p0, sl, s->slots);
            return -1;
        }
        for (int e2 = 0; e2 < e; ++e2)
            if (b->ent_slot[e2] == sl)
            {
                set_error("tllm_stack_step: entries %d and %d share slot %d", e2, e, sl);
                return -1;
            }
        const int nb = (p0 + c + s->page - 1) / s->page;
        if (nb > MB)
        {
            set_error("tllm_stack_step: entry %d needs %d blocks, its table has %d", e, nb, MB);
            return -1;
        }
        for (int j = 0; j < nb; ++j)
        {
            const int id = b->block_table[(size_t) e * MB + j];
            if (id < 0 || id >= s->blocks)
            {
                set_error("tllm_stack_step: entry %d, block %d of its table is %d (pool: %d blocks)", e, j, id, s->blocks);
                return -1;
            }
        }
        sum += c;
        max_count = std::max(max_count, c);
        max_ctx = std::max(max_ctx, p0 + c);
    }
    if (sum != T)
    {
        set_error("tllm_stack_step: the entries hold %lld tokens, the batch %d", (long long) sum, T);
        return -1;
    }
    for (int t = 0; t < T; ++t)
        if (b->tokens[t] < 0 || b->tokens[t] >= s->vocab)
        {
            set_error("tllm_stack_step: token %d at row %d is outside the vocabulary of %d", b->tokens[t], t, s->vocab);
            return -1;
        }
    for (int i = 0; i < NW; ++i)
        if (b->want_rows[i] < 0 || b->want_rows[i] >= T)
        {
            set_error("tllm_stack_step: wanted row %d is outside the batch of %d", b->want_rows[i], T);
            return -1;
        }
    // ---- metadata: one packed int32 image, one copy
    const size_t n_ints = (size_t) 4 * T + (size_t) 5 * E + (size_t) E * MB + NW;
    if (ensure_scratch(s, T, std::max(NW, 1), (int) (n_ints + 3) / 4 * 4))
        return -1;
    const bool deliver = (logits_out || next_ids_out) && ensure_landing(s, NW);
    int32_t* h = s->pinned;
    int32_t *h_tok = h, *h_tent = h + T, *h_tpos = h + 2 * T, *h_first = h + 3 * T, *h_count = h_first + E, *h_pos0 = h_count + E,
            *h_slot = h_pos0 + E, *h_fed = h_slot + E, *h_table = h_fed + E, *h_want = h_table + (size_t) E * MB, *h_prev = h_want + NW;
    std::memcpy(h_tok, b->tokens, (size_t) T * 4);
    int row = 0;
    for (int e = 0; e < E; ++e)
    {
        h_first[e] = row;
        h_count[e] = b->ent_count[e];
        h_pos0[e] = b->ent_pos0[e];
        h_slot[e] = b->ent_slot[e];
        h_fed[e] = b->ent_pos0[e] > 0 ? s->fed[(size_t) b->ent_slot[e]] : 0;
        for (int i = 0; i < b->ent_count[e]; ++i, ++row)
        {
            h_tent[row] = e;
            h_tpos[row] = b->ent_pos0[e] + i;
            // the token before this one in its sequence (-1: none): the row above, or what the slot's sequence ended its last step with
            h_prev[row] = i > 0 ? b->tokens[row - 1] : (b->ent_pos0[e] > 0 ? s->last_tok[(size_t) b->ent_slot[e]] : -1);
        }
        s->last_tok[(size_t) b->ent_slot[e]] = b->tokens[row - 1];
        const int nb = (b->ent_pos0[e] + b->ent_count[e] + s->page - 1) / s->page;
        for (int j = 0; j < MB; ++j)
            h_table[(size_t) e * MB + j] = j < nb ? b->block_table[(size_t) e * MB + j] : 0;
    }
    for (int i = 0; i < NW; ++i)
        h_want[i] = b->want_rows[i];
    const int32_t* d = s->ints;
    const int32_t *d_tok = d, *d_tent = d + T, *d_tpos = d + 2 * T, *d_first = d + 3 * T, *d_count = d_first + E, *d_pos0 = d_count + E,
                  *d_slot = d_pos0 + E, *d_fed = d_slot + E, *d_table = d_fed + E, *d_want = d_table + (size_t) E * MB, *d_prev = d_want + NW;

    const int Wd = s->width;
    const bool looped = s->loop_stop > s->loop_start;
    const int64_t stream_stride = (int64_t) T * Wd;
    StackBegin begin;
    begin.dtype = s->dtype;
    begin.dst = s->ints;
    begin.host = h;
    begin.n = (int) (n_ints + 3) / 4 * 4;
    std::memcpy(begin.ids, h_tok, (size_t) std::min(T, StackBegin::TOKENS) * 4);
    std::memcpy(begin.prev, h_prev, (size_t) std::min(T, StackBegin::TOKENS) * 4);
    begin.x = s->x;
    begin.keep = looped && s->loop_times > 1 ? s->x0 : nullptr;
    begin.table = s->embed;
    begin.pair_table = s->pair_buckets > 0 ? s->pair_table : nullptr;
    begin.tokens = T;
    begin.width = Wd;
    begin.vocab = s->vocab;
    begin.buckets = s->pair_buckets;
    begin.mul_prev = s->pair_mul_prev;
    begin.mul_cur = s->pair_mul_cur;
    begin.copies = s->streams;
    begin.copy_stride = stream_stride;
    begin.scale = s->emb_scale;
    if (!s->plain && stack_begin_serves(begin)) // (a plain residual starts in the launch of its first norm)
    {
        if (launch_stack_begin(begin, stream))
            return -1;
    }
    else if (launch_stack_fetch(begin.dst, begin.host, begin.n, stream)
        || (!s->plain
            && launch_stack_embed(begin.x, begin.keep, d_tok, s->embed, s->dtype, T, Wd, s->vocab, s->emb_scale, stream, s->streams, stream_stride))
        || (s->pair_buckets > 0
            && launch_stack_pair_embed(s->x, d_tok, d_prev, s->pair_table, s->dtype, T, Wd, s->pair_buckets, s->pair_mul_prev, s->pair_mul_cur, stream,
                s->streams, stream_stride)))
        return -1;
    s->tap_tokens = T;

    // P1 = h1 W_mix^T, then the mixer: its context rows land in s->ctx, ld_ctx elements apart
    // first(g): launches it, its row in s->h1 or formed on the way
    StackRowNorm mixed;   // what the out-projection forms ctx from where the mixer left it raw
    bool raw_ctx = false;
    auto run_mixer = [&](const Layer& l, const Run& r, auto first) -> int {
        raw_ctx = false;
        const int64_t ld_ctx = l.n_ctx + (s->side_by_side && l.kind == MIX_LATENT ? l.shared_ff : 0);
        StackGemmParams g;
        g.dtype = s->dtype;
        g.M = T;
        g.N = l.n_mix;
        g.K = Wd;
        g.a = s->h1;
        g.lda = Wd;
        g.w = l.w_mix;
        g.c = s->proj;
        g.ldc = l.n_mix;
        g.bias = l.bias;
        if (s->side_by_side && l.shared_ff > 0)
        {
            GemmSection& sec = g.seam.sec[g.seam.n_sec++];
            sec.col0 = g.N;
            sec.c = l.kind == MIX_LATENT ? (char*) s->ctx + (size_t) l.n_ctx * s->es : (char*) s->act_sh;
            sec.ldc = l.kind == MIX_LATENT ? ld_ctx : l.shared_ff;
            sec.act = ACT_RELU2;
            g.N += l.shared_ff;
        }
        if (l.n_route > 0)
        {
            GemmSection& sec = g.seam.sec[g.seam.n_sec++];
            sec.col0 = g.N;
            sec.c = s->route_z;
            sec.ldc = l.n_route;
            sec.f32 = 1;
            g.N += l.n_route;
        }
        if (first(g))
            return -1;
        if (l.kind == MIX_DELTA)
        {
            // convolution + silu of q | k | v (and the sequence's new tail)
            StackSsmParams sp;
            sp.dtype = s->dtype;
            sp.tokens = T;
            sp.entries = E;
            sp.taps = l.taps;
            sp.proj = s->proj;
            sp.ldp = l.n_mix;
            sp.conv_w = l.conv_w;
            sp.conv_channels = l.n_conv;
            sp.conv_col = 0;
            sp.conv_state = r.conv_state;
            sp.xbc = s->xbc;
            sp.tok_entry = d_tent;
            sp.tok_pos = d_tpos;
            sp.ent_slot = d_slot;
            sp.ent_first = d_first;
            sp.ent_count = d_count;
            sp.ent_pos0 = d_pos0;
            sp.ent_fed = d_fed;
            StackDeltaParams dp;
            dp.max_count = max_count;
            dp.dim = l.dim;
            dp.vdim = l.vdim;
            dp.taps = l.taps;
            dp.conv_w = l.conv_w;
            dp.conv_state = r.conv_state;
            dp.ld_raw = l.n_mix;
            dp.x_raw = stack_delta_convolves(dp) ? s->proj : nullptr;
            if (!dp.x_raw && launch_stack_ssm_conv(sp, stream))
                return -1;
            // the two low-rank projections' second halves, in fp32: the decay's pre-activation and the output gate's
            const int col_b = l.n_conv, col_a = col_b + l.n_beta, col_g = col_a + l.decay_rank;
            StackGemmParams lr;
            lr.dtype = s->dtype;
            lr.out_f32 = 1;
            lr.M = T;
            lr.N = l.heads * l.dim;
            lr.K = l.decay_rank;
            lr.a = (const char*) s->proj + (size_t) col_a * s->es;
            lr.lda = l.n_mix;
            lr.w = l.w_a2;
            lr.c = s->dl_a;
            lr.ldc = lr.N;
            // (a launch instead of two, us: one row, 1024 x 128 3.3 + 3.6, 3.6; 1672 rows 7.7 + 7.7, 13.  Tiles take a pair in one launch where a row is whole stages of 64; rows
            // that end inside one go one by one, by whole stages and a rest, as a pair would
            // not: rank 96, 4 layers of width 1536, 300 rows 690 as pairs and 550 one by one, 2000 rows 1580 and 1470)
            const bool pair = l.low_pair && (T < 32 || l.decay_rank % 64 == 0);
            if (pair)
            {
                lr.batch = 2;
                lr.stride_a = l.decay_rank;
                lr.stride_w = (int64_t) lr.N * lr.K;
                lr.stride_c = s->dl_g - s->dl_a;
            }
            if (launch_stack_gemm(lr, stream))
                return -1;
            lr.N = l.n_ctx;
            lr.K = l.gate_rank;
            lr.a = (const char*) s->proj + (size_t) col_g * s->es;
            lr.w = l.low_pair ? (const char*) l.w_a2 + (size_t) l.n_ctx * l.gate_rank * s->es : l.w_g2;
            lr.c = s->dl_g;
            lr.ldc = lr.N;
            if (!pair && launch_stack_gemm(lr, stream))
                return -1;
            dp.dtype = s->dtype;
            dp.tokens = T;
            dp.entries = E;
            dp.heads = l.heads;
            dp.qk_heads = l.kv_heads;
            dp.x = s->xbc;
            dp.beta_raw = (const char*) s->proj + (size_t) col_b * s->es;
            dp.ld_beta = l.n_mix;
            dp.decay_raw = s->dl_a;
            dp.dt_bias = l.dt_bias;
            dp.a_log = l.a_log;
            dp.gate_raw = s->dl_g;
            dp.norm_w = l.hnorm;
            dp.eps = s->eps;
            dp.state = r.state;
            dp.o32 = s->o32;
            dp.out = s->ctx;
            dp.ent_slot = d_slot;
            dp.ent_first = d_first;
            dp.ent_count = d_count;
            dp.ent_pos0 = d_pos0;
            dp.ent_fed = d_fed;
            dp.chunk_ws = s->chunk_ws;
            dp.chunk_floats = s->chunk_floats;
            return launch_stack_delta(dp, stream);
        }
        if (l.kind == MIX_MAMBA2)
        {
            StackSsmParams sp;
            sp.dtype = s->dtype;
            sp.tokens = T;
            sp.entries = E;
            sp.heads = l.heads;
            sp.vdim = l.vdim;
            sp.state = l.dim;
            sp.groups = l.groups;
            sp.taps = l.taps;
            sp.proj = s->proj;
            sp.ldp = l.n_mix;
            sp.conv_w = l.conv_w;
            sp.conv_b = l.conv_b;
            sp.dt_bias = l.dt_bias;
            sp.a_log = l.a_log;
            sp.d_skip = l.d_skip;
            sp.conv_state = r.conv_state;
            sp.ssm_state = r.state;
            sp.xbc = s->xbc;
            sp.y32 = s->o32;
            sp.tok_entry = d_tent;
            sp.tok_pos = d_tpos;
            sp.ent_slot = d_slot;
            sp.ent_first = d_first;
            sp.ent_count = d_count;
            sp.ent_pos0 = d_pos0;
            sp.ent_fed = d_fed;
            sp.max_count = max_count;
            sp.chunk_ws = s->chunk_ws;
            sp.chunk_floats = s->chunk_floats;
            // convolution + silu (and the sequence's new tail), the recurrence with skip and gate, the norm in parts of the row
            sp.convolve = stack_ssm_convolves(sp);
            if ((!sp.convolve && launch_stack_ssm_conv(sp, stream)) || launch_stack_ssm_scan(sp, stream))
                return -1;
            if (T == 1 && !s->side_by_side && !s->taps)
            {
                // (by the out-projection)
                mixed.x = s->o32;
                mixed.w = l.hnorm;
                mixed.eps = s->eps;
                mixed.parts = l.ssm_norm_groups;
                raw_ctx = stack_row_norm_serves(mixed, s->dtype, l.n_ctx);
                if (raw_ctx)
                    return 0;
            }
            return launch_stack_group_rmsnorm(s->ctx, nullptr, s->o32, nullptr, l.hnorm, nullptr, s->dtype, T, l.n_ctx, l.ssm_norm_groups, s->eps,
                stream);
        }
        if (l.kind == MIX_HGRN2)
        {
            StackHgrnParams hp;
            hp.dtype = s->dtype;
            hp.tokens = T;
            hp.entries = E;
            hp.heads = l.heads;
            hp.dim = l.dim;
            hp.vdim = l.vdim;
            hp.proj = s->proj;
            hp.ldp = l.n_mix;
            hp.f_bias = l.f_bias;
            hp.lower = l.lower;
            hp.norm_w = l.hnorm;
            hp.eps = s->eps;
            hp.state = r.state;
            hp.ent_slot = d_slot;
            hp.ent_first = d_first;
            hp.ent_count = d_count;
            hp.ent_pos0 = d_pos0;
            hp.max_count = max_count;
            hp.chunk_ws = s->chunk_ws;
            hp.chunk_floats = s->chunk_floats;
            hp.o32 = s->o32;
            hp.out = s->ctx;
            return launch_stack_hgrn2(hp, stream);
        }
        StackAttnParams a;
        a.dtype = s->dtype;
        a.tokens = T;
        a.entries = E;
        a.heads = l.heads;
        a.freq = l.freq;
        a.scale = (float) l.scale;
        a.eps = s->eps;
        a.proj = s->proj;
        a.ldp = l.n_mix;
        a.q = s->q;
        a.k_pool = r.k_pool;
        a.v_pool = r.v_pool;
        a.page = s->page;
        a.max_blocks = MB;
        a.block_table = d_table;
        a.tok_entry = d_tent;
        a.tok_pos = d_tpos;
        a.ent_first = d_first;
        a.ent_count = d_count;
        a.ent_pos0 = d_pos0;
        a.max_count = max_count;
        a.max_context = max_ctx;
        a.split_ws = s->attn_ws;
        if (l.kind == MIX_LATENT)
        {
            // absorbed form: one shared key/value head over [latent | rotated part]; queries [W_uk^T q_plain | rotated q part]
            const int C = l.kv_rank, R = l.rot_part, D = l.dim, H = l.heads;
            a.kv_heads = 1;
            a.maps = 1;
            a.dim = C + R;
            a.vdim = C;
            a.rot_dims = l.rot_dims;
            a.rot_halves = l.rot_halves;
            a.mscale = l.mscale;
            a.mask = l.mask;
            a.mask_size = l.mask_size;
            a.sink = l.sinkv;
            if (l.n_gate)
            {
                // the gate scales a head's whole row, so it commutes with the expansion behind the attention
                a.out_gate = (const char*) s->proj + (size_t) (l.n_q + l.n_k + l.n_v + l.n_rg) * s->es;
                a.ld_gate = l.n_mix;
            }
            a.out = s->lat;
            const void* q_src = s->proj;
            int64_t ldq = l.n_mix;
            if (l.q_rank > 0)
            {
                // queries through their own latent: norm of the first q_rank columns, then the expansion to every head's [plain | rotated]
                if (launch_stack_row_rmsnorm(s->cq, l.q_rank, s->proj, l.n_mix, l.cq_norm, s->dtype, T, l.q_rank, s->eps, stream))
                    return -1;
                StackGemmParams uq;
                uq.dtype = s->dtype;
                uq.M = T;
                uq.N = H * (D + R);
                uq.K = l.q_rank;
                uq.a = s->cq;
                uq.lda = l.q_rank;
                uq.w = l.w_uq;
                uq.c = s->qfull;
                uq.ldc = uq.N;
                if (launch_stack_gemm(uq, stream))
                    return -1;
                q_src = s->qfull;
                ldq = uq.N;
            }
            if (launch_stack_latent_prep(a, D, l.lat_norm, stream, q_src, ldq, l.n_q))
                return -1;
            StackGemmParams qa;
            qa.dtype = s->dtype;
            qa.M = T;
            qa.N = C;
            qa.K = D;
            qa.a = q_src;
            qa.lda = ldq;
            qa.w = l.w_ukT;
            qa.c = s->q;
            qa.ldc = (int64_t) H * (C + R);
            qa.batch = H;
            qa.stride_a = D + R;
            qa.stride_w = (int64_t) C * D;
            qa.stride_c = C + R;
            if (launch_stack_gemm(qa, stream) || launch_stack_attention(a, stream))
                return -1;
            StackGemmParams ve; // head h: ctx[:, h] = lat[:, h] W_uv,h^T
            ve.dtype = s->dtype;
            ve.M = T;
            ve.N = l.vdim;
            ve.K = C;
            ve.a = s->lat;
            ve.lda = (int64_t) H * C;
            ve.w = l.w_uv;
            ve.c = s->ctx;
            ve.ldc = ld_ctx;
            ve.batch = H;
            ve.stride_a = C;
            ve.stride_w = (int64_t) l.vdim * C;
            ve.stride_c = l.vdim;
            return launch_stack_gemm(ve, stream);
        }
        a.kv_heads = l.kv_heads;
        a.maps = l.maps;
        a.dim = l.dim;
        a.vdim = l.vdim;
        a.rot_dims = l.rot_dims;
        a.rot_halves = l.rot_halves;
        a.mscale = l.mscale;
        a.softcap = (float) l.softcap;
        a.lambda = l.lambda;
        a.out_scale = (float) (1.0 - l.diff);
        a.head_norm = l.head_norm;
        a.temp = l.temp;
        a.slope = l.slope;
        a.log_r1 = l.r1;
        a.log_r2 = l.r2;
        a.mask = l.mask;
        a.mask_size = l.mask_size;
        a.mask_keep = l.mask_keep;
        a.talk = l.talkw;
        a.pair_ws = l.talk ? s->pairs : nullptr;
        if (l.v_mix)
        {
            a.v_first = s->v_first;
            a.v_first_write = r.layer == s->v_mix_first;
            a.v_mix = l.vmix;
        }
        a.values_are_keys = l.values_are_keys;
        a.gate_wide = l.gate_wide;
        a.q_norm_w = l.q_norm;
        a.k_norm_w = l.k_norm;
        a.weights = l.weights;
        a.sink = l.sinkv;
        a.wbias = l.wbias;
        a.qk_unit_norm = l.qk_norm;
        if (l.n_gate)
        {
            a.out_gate = (const char*) s->proj + (size_t) (l.n_q + l.n_k + l.n_v + l.n_rg) * s->es;
            a.ld_gate = l.n_mix;
        }
        a.out = s->ctx;
        return (launch_stack_rope_kv(a, stream) || launch_stack_attention(a, stream)) ? -1 : 0;
    };

    // the routed feed-forward on h1: y = its output, or (accumulate) y += it, x_el = the resulting rows in the element type; later != null: what y
    // stands for, for the norm that reads it.  With residual=plain the router's logits are there already.  form(mp): h1 is still to be formed, by a launch of its own
    // or (mp != null) by the one of mp's logits; 1: those are there.
    auto run_moe = [&](const Layer& l, float* y, bool accumulate, void* y_el, StackExpertSum* later, auto form) -> int {
        const size_t pairs = (size_t) T * l.top;
        StackMoeParams mp;
        mp.dtype = s->dtype;
        mp.tokens = T;
        mp.width = Wd;
        mp.experts = l.experts;
        mp.identity = l.identity;
        mp.top = l.top;
        mp.group_count = l.route_groups;
        mp.group_keep = l.route_keep;
        mp.scale = (float) l.route_scale;
        mp.score = l.route_sigmoid ? ROUTE_SIGMOID : ROUTE_SOFTMAX;
        mp.weight_input = l.route_weight_input;
        mp.normalize = l.route_norm;
        mp.h = s->h1;
        mp.router_w = l.router_w;
        mp.correction = l.correction;
        mp.bias = l.route_b;
        mp.topk_idx = s->moe_i;
        mp.slot_of_pair = s->moe_i + pairs;
        mp.pair_of_slot = s->moe_i + 2 * pairs;
        mp.tok_of_slot = s->moe_i + 3 * pairs;
        mp.group_off = s->moe_i + 4 * pairs;
        mp.topk_w = s->moe_w;
        mp.logits = s->plain ? s->route_z : s->moe_w + pairs;
        mp.have_logits = s->plain ? 1 : 0;
        mp.ticket = s->moe_ticket;
        mp.a_sorted = l.route_weight_input ? s->moe_a : nullptr; // otherwise the products read h1 through the slots' tokens
        mp.accumulate = accumulate ? 1 : 0;
        mp.accumulate_gate = l.shared_gate ? s->shared_z : nullptr;
        mp.y_el = y_el;
        // per expert: gate and up on its rows with silu(gate) * up (or relu(up)^2) in the epilogue, down in fp32; an expert's rows are at most one per token
        const int up_cols = l.expert_relu2 ? l.ff : 2 * l.ff;
        StackGemmParams u;
        u.dtype = s->dtype;
        u.M = T;
        u.N = up_cols;
        u.K = Wd;
        u.a = mp.a_sorted ? s->moe_a : s->h1;
        u.a_rows = mp.a_sorted || T == 1 ? nullptr : mp.tok_of_slot;
        u.lda = mp.a_sorted || T > 1 ? Wd : 0; // (every slot of a lone token reads its row: nothing to look up)
        u.w = l.w_gu;
        u.c = s->act;
        u.ldc = l.ff;
        u.act = l.expert_relu2 ? ACT_RELU2 : ACT_GATE_SILU;
        u.batch = l.experts;
        u.stride_w = (int64_t) up_cols * Wd;
        u.group_off = mp.group_off;
        u.group_total = (int) pairs;
        u.group_rows = (int) std::min<int64_t>(T, (pairs + l.experts + l.identity - 1) / (l.experts + l.identity)); // (identity experts' choices are no rows)
        StackGemmParams dn;
        dn.dtype = s->dtype;
        dn.out_f32 = 1;
        dn.M = T;
        dn.N = Wd;
        dn.K = l.ff;
        dn.a = s->act;
        dn.lda = l.ff;
        dn.w = l.w_down;
        dn.c = s->moe_y;
        dn.ldc = Wd;
        dn.batch = l.experts;
        dn.stride_w = (int64_t) Wd * l.ff;
        dn.group_off = mp.group_off;
        dn.group_total = u.group_total;
        dn.group_rows = u.group_rows;
        StackGemmParams lone = u; // (reads the token's row itself, also where it counts weighted)
        lone.a = s->h1;
        const bool choosing = stack_lone_serves(mp, lone, dn);
        const int formed = form(choosing && !mp.have_logits ? &mp : nullptr);
        if (formed < 0)
            return -1;
        if (choosing)
        {
            if ((!mp.have_logits && !formed && launch_stack_moe_logits(mp, stream)) || launch_stack_lone_up(mp, lone, stream) || launch_stack_lone_down(mp, dn, stream))
                return -1;
        }
        else if (launch_stack_moe_plan(mp, stream) || launch_stack_gemm(u, stream) || launch_stack_gemm(dn, stream))
            return -1;
        // (in the norm one workgroup forms a row's sum: few tokens with very many choices are better off with the combining launch, which spreads a row.
        // A layer's norms and sum, us, in the norm / apart: 64 rows of 6144, 1 token 31.4 / 27.6, 8 33.4 / 28.5, 64 36.4 / 33.3, 128 42 either way; 32 rows of
        // 6144 21.0 / 20.0, 23.0 / 22.1, 26.0 / 26.1)
        if (!later || (T <= 64 && (int64_t) l.top * Wd > 128 * 1024))
            return launch_stack_moe_combine(mp, s->moe_y, y, stream);
        later->ys = s->moe_y;
        later->slot_of_pair = mp.slot_of_pair;
        later->topk_w = mp.topk_w;
        later->h = mp.h;
        later->keep = mp.accumulate_gate;
        later->tokens = T;
        later->top = l.top;
        later->weight_input = mp.weight_input;
        later->has_row = mp.accumulate;
        return 0;
    };

    StackExpertSum left_sum; // what y32 stands for where the last sublayer was a mixture of experts

    auto product = [&](const StackGemmParams& g) { return launch_stack_gemm(g, stream); };
    auto formed_before = [](const StackMoeParams*) { return 0; };
    // a layer's out-projection, behind its mixer
    auto out_product = [&](const StackGemmParams& g) -> int {
        if (raw_ctx)
        {
            const int rc = launch_stack_row_gemm(g, mixed, stream);
            if (rc <= 0)
                return rc;
            if (launch_stack_group_rmsnorm(s->ctx, nullptr, mixed.x, nullptr, mixed.w, nullptr, s->dtype, T, g.K, mixed.parts, mixed.eps, stream))
                return -1;
        }
        return launch_stack_gemm(g, stream);
    };

    // the feed-forwards of sequential blocks: h1 -> y32
    auto seq_dense = [&](const Layer& l, auto first) -> int {
        StackGemmParams u;
        u.dtype = s->dtype;
        u.M = T;
        u.K = Wd;
        u.a = s->h1;
        u.lda = Wd;
        u.w = l.w_gu;
        u.N = l.mlp == MLP_RELU2 ? l.ff : 2 * l.ff;
        u.c = s->act;
        u.ldc = l.ff;
        u.act = l.mlp == MLP_RELU2 ? ACT_RELU2 : ACT_GATE_GELU;
        if (first(u))
            return -1;
        StackGemmParams dn;
        dn.dtype = s->dtype;
        dn.out_f32 = 1;
        dn.M = T;
        dn.N = Wd;
        dn.K = l.ff;
        dn.a = s->act;
        dn.lda = l.ff;
        dn.w = l.w_down;
        dn.c = s->y32;
        dn.ldc = Wd;
        return launch_stack_gemm(dn, stream);
    };
    auto seq_moe = [&](const Layer& l, auto form) -> int {
        // what reads the row beside the experts, one product: the shared expert's first matrices, with residual=plain the router's logits,
        // the shared expert's gate (both in fp32)
        const int n_z = s->plain ? l.experts + l.identity : 0;
        const bool alone = l.n_shared + n_z == 0; // nothing but the routed layer reads h1
        if (!alone && form(nullptr) < 0)
            return -1;
        StackGemmParams u;
        u.dtype = s->dtype;
        u.M = T;
        u.N = l.n_shared;
        u.K = Wd;
        u.a = s->h1;
        u.lda = Wd;
        u.w = l.w_shared_up;
        u.c = s->act_sh;
        u.ldc = l.shared_ff;
        u.act = l.expert_relu2 ? ACT_RELU2 : ACT_GATE_SILU;
        if (l.n_shared == 0)
        {
            u.N = n_z;
            u.c = s->route_z;
            u.ldc = n_z;
            u.out_f32 = 1;
            u.act = ACT_NONE;
        }
        else
        {
            auto section = [&](float* c, int n) {
                GemmSection& sec = u.seam.sec[u.seam.n_sec++];
                sec.col0 = u.N;
                sec.c = c;
                sec.ldc = n;
                sec.f32 = 1;
                u.N += n;
            };
            if (n_z > 0)
                section(s->route_z, n_z);
            if (l.shared_gate)
                section(s->shared_z, 1);
        }
        if (u.N > 0 && launch_stack_gemm(u, stream))
            return -1;
        if (l.shared_ff > 0)
        {
            StackGemmParams sd;
            sd.dtype = s->dtype;
            sd.out_f32 = 1;
            sd.M = T;
            sd.N = Wd;
            sd.K = l.shared_ff;
            sd.a = s->act_sh;
            sd.lda = l.shared_ff;
            sd.w = l.w_shared_down;
            sd.c = s->y32;
            sd.ldc = Wd;
            if (launch_stack_gemm(sd, stream))
                return -1;
        }
        return run_moe(l, s->y32, l.shared_ff > 0, nullptr, &left_sum, [&](const StackMoeParams* mp) { return alone ? form(mp) : 0; });
    };

    // residual=plain: what the last sublayer or token input left to land in y32, and the next norm, in one launch
    bool land_y = false;              // y32 holds a result that is not in x yet
    const float* land_norm = nullptr; // weight of the norm on it, null: as it is
    auto land = [&](void* h, const float* w, const float* add_row, const int32_t* rows, int n, float* tap, bool start) -> int {
        StackLandParams lp;
        lp.dtype = s->dtype;
        lp.tokens = n;
        lp.width = Wd;
        lp.x = s->x;
        if (start)
        {
            lp.table = s->embed;
            lp.ids = d_tok;
            lp.vocab = s->vocab;
            lp.scale = s->emb_scale;
            lp.y_norm = s->embed_norm_w;
        }
        else if (land_y)
        {
            lp.y = s->y32;
            lp.sum = left_sum;
            lp.y_norm = land_norm;
            lp.y_scale = s->resid_mult;
        }
        lp.tap = tap;
        lp.add_row = add_row;
        lp.h = h;
        lp.w = w;
        lp.eps = s->eps;
        lp.rows = rows;
        land_y = false;
        land_norm = nullptr;
        left_sum = StackExpertSum();
        return launch_stack_land(lp, stream);
    };

    // residual=hyper: the sublayer result in y32 that has not yet been folded into the streams, and the launch that folds it,
    // combines the streams for the next reader and norms the combination
    const HyperW* pending = nullptr;
    float* xs = s->x; // the streams; a lone token's single one changes places with x0 where a launch folds a result in that others read at the same time
    auto hyper_of = [&](const float* in, void* h, const float* w, float* sum_out) -> StackHyperParams {
        StackHyperParams hp;
        hp.dtype = s->dtype;
        hp.tokens = T;
        hp.width = Wd;
        hp.streams = s->streams;
        hp.x = xs;
        hp.stream_stride = stream_stride;
        if (pending)
        {
            hp.y = s->y32;
            hp.sum = left_sum;
            hp.mix = pending->mix;
            hp.out = pending->out;
        }
        hp.in = in;
        hp.h = h;
        hp.w = w;
        hp.eps = s->eps;
        hp.sum_out = sum_out;
        return hp;
    };
    auto hyper_norm = [&](const StackHyperParams& hp) -> int {
        pending = nullptr;
        left_sum = StackExpertSum();
        return launch_stack_hyper_norm(hp, stream);
    };
    auto hyper = [&](const float* in, void* h, const float* w, float* sum_out) { return hyper_norm(hyper_of(in, h, w, sum_out)); };

    // A lone token's normed row is formed by the launch that reads it, launch(row), where that is the only one, or the first and leaves it for the others; 1: it is not.
    // (what waits for the stream as a sum of experts is formed once, by the norm's own launch; with taps every norm has one, here and below)
    auto lone_row = [&](const float* in, const float* w, void* h, auto launch) -> int {
        if (T != 1 || !s->hyper || s->streams != 1 || s->taps || (pending && left_sum.ys))
            return 1;
        StackRowNorm n;
        n.x = xs;
        if (pending)
        {
            n.y = s->y32;
            n.mix = pending->mix;
            n.out = pending->out;
            n.x_out = xs == s->x ? s->x0 : s->x;
        }
        n.in = in;
        n.w = w;
        n.eps = s->eps;
        n.h = h;
        const int rc = launch(n);
        if (rc == 0)
        {
            xs = pending ? n.x_out : xs;
            pending = nullptr;
        }
        return rc;
    };

    for (size_t ri = 0; ri < s->runs.size(); ++ri)
    {
        const Run& r = s->runs[ri];
        const Layer& l = s->layers[r.layer];
        if (s->side_by_side)
        {
            if (land(s->h1, l.norm1, r.enters_pass ? s->loop_step + (size_t) r.pass * Wd : nullptr, nullptr, T,
                    s->taps && ri > 0 ? s->tap + (ri - 1) * (size_t) T * Wd : nullptr, ri == 0))
                return -1;
            if (run_mixer(l, r, product))
                return -1;
            const bool joint = l.kind == MIX_LATENT && l.shared_ff > 0;
            StackGemmParams o; // x += [ctx | a_shared] [Wo | Wshared_down]^T
            o.dtype = s->dtype;
            o.M = T;
            o.N = Wd;
            o.K = l.n_ctx + (joint ? l.shared_ff : 0);
            o.a = s->ctx;
            o.lda = o.K;
            o.w = l.w_o;
            o.resid = s->x;
            o.ldr = Wd;
            if (launch_stack_gemm(o, stream))
                return -1;
            if (l.shared_ff > 0 && !joint)
            {
                o.K = l.shared_ff;
                o.a = s->act_sh;
                o.lda = o.K;
                o.w = l.w_shared_down;
                if (launch_stack_gemm(o, stream))
                    return -1;
            }
            if (l.ff > 0 && run_moe(l, s->x, true, s->side_dim ? s->x_el : nullptr, nullptr, formed_before))
                return -1;
            if (s->side_dim > 0)
            {
                if (l.ff == 0 && land(s->x_el, nullptr, nullptr, nullptr, T, nullptr, false))
                    return -1;
                StackGemmParams sg; // g = gelu(Wgate x) * the layer's part of the token's side embedding
                sg.dtype = s->dtype;
                sg.M = T;
                sg.N = s->side_dim;
                sg.K = Wd;
                sg.a = s->x_el;
                sg.lda = Wd;
                sg.w = l.side_gate;
                sg.c = s->side_act;
                sg.ldc = s->side_dim;
                sg.split_ws = s->split_ws;
                sg.split_floats = (int64_t) s->cap_tokens * s->side_dim * kSideParts;
                sg.act = ACT_GELU_MUL;
                sg.seam.mul = (const char*) s->side_embed + (size_t) r.layer * s->side_dim * s->es;
                sg.seam.mul_rows = d_tok;
                sg.seam.ld_mul = (int64_t) s->side_dim * (int64_t) s->layers.size();
                StackGemmParams sp;
                sp.dtype = s->dtype;
                sp.out_f32 = 1;
                sp.M = T;
                sp.N = Wd;
                sp.K = s->side_dim;
                sp.a = s->side_act;
                sp.lda = s->side_dim;
                sp.w = l.side_proj;
                sp.c = s->y32;
                sp.ldc = Wd;
                if (launch_stack_gemm(sg, stream) || launch_stack_gemm(sp, stream))
                    return -1;
                land_y = true;
                land_norm = l.side_norm;
            }
            continue;
        }
        if (s->sequential)
        {
            if (s->plain)
            {
                if (land(s->h1, l.norm1, r.enters_pass ? s->loop_step + (size_t) r.pass * Wd : nullptr, nullptr, T,
                        s->taps && ri > 0 ? s->tap + (ri - 1) * (size_t) T * Wd : nullptr, ri == 0))
                    return -1;
            }
            else if (s->token_shift)
            {
                // the mixer reads the normed row blended with the previous token's: in the norm's launch, or of rows that it leaves in fp32
                StackHyperParams hp = hyper_of(l.hc[0].in, s->h1, l.norm1, nullptr);
                hp.mu = l.shift;
                hp.carry = r.shift_carry;
                hp.ent_slot = d_slot;
                hp.ent_pos0 = d_pos0;
                const bool together = max_count == 1 && stack_hyper_shifts(hp);
                if (!together)
                {
                    hp.carry = nullptr;
                    hp.h = nullptr;
                    hp.h32 = s->h32;
                }
                if (hyper_norm(hp))
                    return -1;
                if (!together)
                {
                    StackShiftParams sh;
                    sh.dtype = s->dtype;
                    sh.tokens = T;
                    sh.entries = E;
                    sh.width = Wd;
                    sh.n = s->h32;
                    sh.mu = l.shift;
                    sh.carry = r.shift_carry;
                    sh.h = s->h1;
                    sh.tok_entry = d_tent;
                    sh.tok_pos = d_tpos;
                    sh.ent_slot = d_slot;
                    sh.ent_first = d_first;
                    sh.ent_count = d_count;
                    sh.ent_pos0 = d_pos0;
                    if (launch_stack_token_shift(sh, stream))
                        return -1;
                }
            }
            // a sublayer's result waits in y32 for the next launch that reads the stream
            auto leave = [&](int sub) {
                pending = &l.hc[sub];
                land_y = true;
                land_norm = sub ? l.norm2b : l.norm1b;
            };
            // g reads the row that norm1 or norm2 forms; with residual=plain and behind a token shift it is there
            auto normed = [&](const StackGemmParams& g, int sub) -> int {
                const float *in = l.hc[sub].in, *w = sub ? l.norm2 : l.norm1;
                if (!s->plain && !(s->token_shift && sub == 0))
                {
                    const int rc = lone_row(in, w, nullptr, [&](const StackRowNorm& n) { return launch_stack_row_gemm(g, n, stream); });
                    if (rc <= 0)
                        return rc;
                    if (hyper(in, s->h1, w, nullptr))
                        return -1;
                }
                return launch_stack_gemm(g, stream);
            };
            if (run_mixer(l, r, [&](const StackGemmParams& g) { return normed(g, 0); }))
                return -1;
            StackGemmParams o; // y = ctx Wo^T in fp32: the residual sum is 32-bit
            o.dtype = s->dtype;
            o.out_f32 = 1;
            o.M = T;
            o.N = Wd;
            o.K = l.n_ctx;
            o.a = s->ctx;
            o.lda = l.n_ctx;
            o.w = l.w_o;
            o.c = s->y32;
            o.ldc = Wd;
            o.bias = l.o_biasv;
            if (out_product(o))
                return -1;
            leave(0);
            if (l.ff > 0)
            {
                if (s->plain && land(s->h1, l.norm2, nullptr, nullptr, T, nullptr, false))
                    return -1;
                auto form = [&](const StackMoeParams* mp) -> int {
                    if (s->plain)
                        return 0;
                    const int rc = mp ? lone_row(l.hc[1].in, l.norm2, s->h1, [&](const StackRowNorm& n) {
                        return stack_row_norm_serves(n, s->dtype, Wd) ? launch_stack_moe_logits(*mp, n, stream) : 1;
                    }) : 1;
                    return rc <= 0 ? (rc == 0 ? 1 : -1) : hyper(l.hc[1].in, s->h1, l.norm2, nullptr);
                };
                if (l.mlp == MLP_MOE ? seq_moe(l, form) : seq_dense(l, [&](const StackGemmParams& g) { return normed(g, 1); }))
                    return -1;
                leave(1);
            }
            if (s->hyper && s->taps && hyper(nullptr, nullptr, nullptr, s->tap + ri * (size_t) T * Wd))
                return -1;
            continue;
        }
        if (r.enters_pass
            && launch_stack_pass_entry(s->x, r.pass > 0 ? s->x0 : nullptr, s->loop_step + (size_t) r.pass * Wd, T, Wd, stream))
            return -1;
        auto normed = [&](const StackGemmParams& g) -> int {
            if (T == 1 && !s->taps)
            {
                StackRowNorm n;
                n.x = s->x;
                n.w = l.norm1;
                n.w2 = l.norm2;
                n.h2 = l.ff > 0 ? s->h2 : nullptr;
                n.eps = s->eps;
                n.parts = s->groups;
                const int rc = launch_stack_row_gemm(g, n, stream);
                if (rc <= 0)
                    return rc;
            }
            return launch_stack_group_rmsnorm(s->h1, l.ff > 0 ? s->h2 : nullptr, s->x, nullptr, l.norm1, l.norm2, s->dtype, T, Wd, s->groups, s->eps, stream)
                    || launch_stack_gemm(g, stream)
                ? -1
                : 0;
        };
        if (run_mixer(l, r, normed))
            return -1;
        // x += sigmoid(P1[rg1] + b1) * (ctx Wo^T)
        StackGemmParams o;
        o.dtype = s->dtype;
        o.M = T;
        o.N = Wd;
        o.K = l.n_ctx;
        o.a = s->ctx;
        o.lda = l.n_ctx;
        o.w = l.w_o;
        o.resid = s->x;
        o.ldr = Wd;
        o.gate = (const char*) s->proj + (size_t) (l.n_q + l.n_k + l.n_v) * s->es;
        o.ldg = l.n_mix;
        o.gate_bias = l.rg1_b;
        if (out_product(o))
            return -1;
        if (l.ff > 0)
        {
            // the feed-forward reads the same x as the mixer (h2 was normed before the mixer's update landed); P1's columns are
            // consumed once the mixer and the O product have run, so P2 may take their place
            StackGemmParams u;
            u.dtype = s->dtype;
            u.M = T;
            u.K = Wd;
            u.a = s->h2;
            u.lda = Wd;
            u.w = l.w_gu;
            u.c = s->act;
            u.ldc = l.ff;
            u.act = ACT_GATE_GELU;
            u.N = 2 * l.ff + Wd;
            u.seam.n_sec = 1; // the residual gate's columns
            u.seam.sec[0].col0 = 2 * l.ff;
            u.seam.sec[0].c = s->proj;
            u.seam.sec[0].ldc = Wd;
            if (launch_stack_gemm(u, stream))
                return -1;
            StackGemmParams dn;
            dn.dtype = s->dtype;
            dn.M = T;
            dn.N = Wd;
            dn.K = l.ff;
            dn.a = s->act;
            dn.lda = l.ff;
            dn.w = l.w_down;
            dn.resid = s->x;
            dn.ldr = Wd;
            dn.gate = s->proj;
            dn.ldg = Wd;
            dn.gate_bias = l.rg2_b;
            if (launch_stack_gemm(dn, stream))
                return -1;
        }
        if (s->taps)
            HIP_OK(hipMemcpyAsync(s->tap + ri * (size_t) T * Wd, s->x, (size_t) T * Wd * 4, hipMemcpyDeviceToDevice, stream));
    }
    if (s->plain && s->taps && land(nullptr, nullptr, nullptr, nullptr, T, s->tap + (s->runs.size() - 1) * (size_t) T * Wd, false))
        return -1;
    if (NW > 0)
    {
        if (s->plain)
        {
            // the output norm, on the wanted rows only; what the last layer left lands in the same launch
            if (land(s->hw, s->final_norm, nullptr, d_want, NW, nullptr, false))
                return -1;
        }
        else if (s->hyper)
        {
            // the output norm reads the sum of the streams; the last sublayer lands in the same launch, on the wanted rows only
            StackHyperParams hp;
            hp.dtype = s->dtype;
            hp.tokens = NW;
            hp.width = Wd;
            hp.streams = s->streams;
            hp.x = xs;
            hp.stream_stride = stream_stride;
            if (pending)
            {
                hp.y = s->y32;
                hp.sum = left_sum;
                hp.mix = pending->mix;
                hp.out = pending->out;
            }
            hp.h = s->hw;
            hp.w = s->final_norm;
            hp.eps = s->eps;
            hp.rows = d_want;
            if (launch_stack_hyper_norm(hp, stream))
                return -1;
        }
        else if (launch_stack_group_rmsnorm(s->hw, nullptr, s->x, d_want, s->final_norm, nullptr, s->dtype, NW, Wd, s->groups, s->eps, stream))
            return -1;
        StackGemmParams hd;
        hd.dtype = s->dtype;
        hd.out_f32 = 1;
        hd.M = NW;
        hd.N = s->vocab;
        hd.K = Wd;
        hd.a = s->hw;
        hd.lda = Wd;
        hd.w = s->head;
        hd.c = s->logits;
        hd.ldc = s->vocab;
        if (s->logit_scale != 1.f || s->logit_cap > 0.f)
        {
            hd.act = ACT_SCALE_CAP;
            hd.seam.act_scale = s->logit_scale;
            hd.seam.act_cap = s->logit_cap;
        }
        if (launch_stack_gemm(hd, stream))
            return -1;
        if (deliver)
            std::fill_n(s->land_choice, (size_t) NW * stack_choice_parts(s->vocab), stack_no_choice);
        if (deliver && (logits_out || next_ids_out)
            && launch_stack_deliver(logits_out ? s->land_rows : nullptr, s->land_choice, s->logits, NW, s->vocab, stream))
            return -1;
        if (!deliver && next_ids_out && launch_argmax(s->ids_out, s->logits, NW, s->vocab, stream))
            return -1;
        if (!deliver && logits_out)
            HIP_OK(hipMemcpyAsync(logits_out, s->logits, (size_t) NW * s->vocab * 4, hipMemcpyDeviceToHost, stream));
        if (!deliver && next_ids_out)
            HIP_OK(hipMemcpyAsync(next_ids_out, s->ids_out, (size_t) NW * 4, hipMemcpyDeviceToHost, stream));
    }
    if (deliver && logits_out)
        bring_in(logits_out, (size_t) NW * s->vocab * 4);
    const int there = deliver && lands_soon(s, T) ? copy_as_they_land(logits_out, s->land_rows, s->land_choice, NW, s->vocab) : 0; // rows
    if (!deliver || there < NW || s->taps)
        HIP_OK(hipStreamSynchronize(stream));
    if (deliver && logits_out && there < NW)
        std::memcpy(logits_out + (size_t) there * s->vocab, s->land_rows + (size_t) there * s->vocab, (size_t) (NW - there) * s->vocab * 4);
    if (deliver && next_ids_out)
    {
        const int parts = stack_choice_parts(s->vocab);
        for (int i = 0; i < NW; ++i)
            next_ids_out[i] = stack_choose(s->land_choice + (size_t) i * parts, parts);
    }
    for (int e = 0; e < E; ++e)
    {
        constexpr int FAR = 1 << 30, TURNS = FAR / 720720 * 720720; // (whole turns of a ring of up to 16 rows)
        const int rows = h_fed[e] + b->ent_count[e];
        s->fed[(size_t) b->ent_slot[e]] = rows < FAR ? rows : rows - TURNS;
    }
    return 0;
}

int32_t tllm_stack_page_size(tllm_stack_t s)
{
    return s ? s->page : 0;
}
int32_t tllm_stack_num_blocks(tllm_stack_t s)
{
    return s ? s->blocks : 0;
}
int32_t tllm_stack_num_slots(tllm_stack_t s)
{
    return s ? s->slots : 0;
}
int32_t tllm_stack_vocab(tllm_stack_t s)
{
    return s ? s->vocab : 0;
}
int32_t tllm_stack_layer_runs(tllm_stack_t s)
{
    return s ? (int32_t) s->runs.size() : 0;
}
int64_t tllm_stack_weight_bytes(tllm_stack_t s)
{
    return s ? s->weight_bytes : 0;
}

int64_t tllm_stack_step_bytes(tllm_stack_t s, int32_t n_tokens, int64_t context_tokens, int32_t n_entries)
{
    if (!s)
        return 0;
    // weights once (a looped layer's weights once per pass), keys and values of the contexts once per attention run, states read and
    // written once per recurrent run, the embedding rows instead of the whole table
    int64_t bytes = (int64_t) s->vocab * s->width * s->es + (int64_t) n_tokens * s->width * s->es;
    for (const Run& r : s->runs)
    {
        const Layer& l = s->layers[r.layer];
        int64_t ff_rows = l.ff > 0 ? (l.mlp == MLP_RELU2 || l.expert_relu2 ? 2 : 3) * (int64_t) l.ff + l.n_rg : 0;
        if (l.ff > 0 && l.mlp == MLP_MOE)
        {
            // the experts that the step's tokens can reach at most, and the fp32 router
            ff_rows *= std::min<int64_t>(l.experts, (int64_t) n_tokens * l.top);
            bytes += (int64_t) (l.experts + l.identity) * s->width * (s->plain ? s->es : 4);
            ff_rows += (l.expert_relu2 ? 2 : 3) * (int64_t) l.shared_ff + l.shared_gate;
        }
        bytes += 2 * (int64_t) s->side_dim * s->width * s->es + (int64_t) n_tokens * s->side_dim * s->es; // the token input
        bytes += ((int64_t) l.n_mix + l.n_ctx + ff_rows) * s->width * s->es;
        if (l.kind == MIX_LATENT && l.q_rank > 0)
            bytes += (int64_t) l.heads * (l.dim + l.rot_part) * l.q_rank * s->es;
        if (l.kind == MIX_LATENT)
        {
            // the two per-head expansions, and per context token the key row [latent | rotated part] and the latent again as value
            bytes += (int64_t) l.heads * l.kv_rank * (l.dim + l.vdim) * s->es;
            const int64_t ctx = l.mask == MASK_CAUSAL ? context_tokens : std::min<int64_t>(context_tokens, (int64_t) n_entries * l.mask_size);
            bytes += ctx * (2 * (int64_t) l.kv_rank + l.rot_part) * s->es;
        }
        else if (l.kind == MIX_ATTENTION)
        {
            // a window or a chunk bounds what a row reads of its context
            const int64_t ctx = l.mask == MASK_CAUSAL ? context_tokens : std::min<int64_t>(context_tokens, (int64_t) n_entries * l.mask_size);
            bytes += ctx * ((int64_t) l.n_k + l.n_v) * s->es;
        }
        else if (l.kind == MIX_DELTA)
            bytes += ((int64_t) l.heads * l.dim * l.decay_rank + (int64_t) l.n_ctx * l.gate_rank) * s->es
                + 2 * (int64_t) n_entries * ((int64_t) l.heads * l.dim * l.vdim + (int64_t) (l.taps - 1) * l.n_conv) * 4;
        else if (l.kind == MIX_MAMBA2)
            bytes += 2 * (int64_t) n_entries * ((int64_t) l.heads * l.dim * l.vdim + (int64_t) (l.taps - 1) * l.n_conv) * 4;
        else
            bytes += 2 * (int64_t) n_entries * l.heads * l.dim * l.vdim * 4;
    }
    return bytes;
}

int32_t tllm_stack_get_tap(tllm_stack_t s, int32_t run, float* out, size_t n_floats)
{
    if (!s || !s->taps || !s->tap || run < 0 || run >= (int) s->runs.size() || n_floats != (size_t) s->tap_tokens * s->width)
    {
        set_error("tllm_stack_get_tap: taps are off (debug_taps=1), or run / size do not fit the last step");
        return -1;
    }
    HIP_OK(hipMemcpy(out, s->tap + (size_t) run * s->tap_tokens * s->width, n_floats * 4, hipMemcpyDeviceToHost));
    return 0;
}

void tllm_stack_destroy(tllm_stack_t s)
{
    delete s;
}

} // extern "C"
