"""The work that users of this framework have it do, as cases that a timing program can prepare, run and check.

Two engines serve requests here.  `NativeSession` runs LLaMA on a rectangular batch (fp16, SmoothQuant int8, weight-only int8 and int4 weights),
`RaggedGenerationSession` runs the stack designs in packed steps.  A pass is one whole request, or one batch of them, the way a server
issues it: the prompt phase and the generation steps behind it, with nothing kept from the pass before.  The engine with its weights
belongs to the program and outlives its requests, so cases that run on the same engine share one; the prompts come from the seed.

A LLaMA case is {path: llama, mode, width, layers, batch, prompt, new, ragged}: `batch` prompts of up to `prompt` tokens (all of that
length, or from half of it on where `ragged`), `new` tokens generated behind each; 0: the prompt phase and its logits alone.
A stack case is {path: tolenex | rofozen | narurax | ruzinex, width, layers, batch, prompt, new, ragged}: the prompts are fed in steps of
at most 2048 tokens, then every request takes `new` single tokens that are already known (a recorded answer is scored), the logits of
every one of them come back; 0: the logits of the prompt's last four places."""
import gc
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.realpath(__file__)))
sys.path.insert(0, os.path.join(ROOT, 'trtllm-llama_amd'))

VOCAB = 32000
BUDGET = 2048  # tokens of one step, RaggedGenerationSession's own default
QUANT_MODE = {'fp16': 0, 'woq4': 1 | 32, 'woq8': 2 | 32, 'sq': 2 | 4 | 8 | 32}  # every quantised form keeps its cache in int8
STACKS = ('tolenex', 'rofozen', 'narurax', 'ruzinex')


# ------------------------------------------------------------------------------------------------------------------ the cases
def _llama(name, mode, layers, batch, prompt, new, ragged=False, width=4096):
    return dict(name=name, path='llama', mode=mode, width=width, layers=layers, batch=batch, prompt=prompt, new=new, ragged=ragged)


def _stack(name, path, width, batch, prompt, new, ragged=False, layers=4):
    return dict(name=name, path=path, width=width, layers=layers, batch=batch, prompt=prompt, new=new, ragged=ragged)


def listed():
    return [
        # the headline: LLaMA-7B in int8 answers one user behind a 1024-token context
        _llama('llama_sq_chat', 'sq', 32, 1, 1024, 24),
        # an unquantised model, several users, prompts of different lengths (padded rows, masked slots)
        _llama('llama_fp16_batch', 'fp16', 32, 4, 300, 12, ragged=True),
        # weight-only int8: a short question, where generation is nearly all of the time
        _llama('llama_woq8_short', 'woq8', 32, 1, 19, 24),
        # long documents read, for the logits behind them: the matrix products at their largest
        _llama('llama_sq_documents', 'sq', 32, 2, 2048, 0),
        # a small model and a tiny question: latency and launches count
        _llama('llama_small_call', 'fp16', 4, 1, 7, 4, width=1024),
        # a 1024-token prompt through attention and HGRN2 layers
        _stack('tolenex_prompt', 'tolenex', 2048, 1, 1024, 0),
        # state-space, latent-attention and routed layers: a prompt of an odd length and an answer
        _stack('rofozen_chat', 'rofozen', 2048, 1, 1021, 24),
        # delta-rule layers, head-mixed attention, routed layers: prompts of several users in one packed step
        _stack('narurax_prompts', 'narurax', 2048, 3, 683, 0, ragged=True),
        # grouped-query attention, dense and routed feed-forwards at the width of a 7B model: the longest prompt
        _stack('ruzinex_long', 'ruzinex', 4096, 1, 4096, 0),
        # eight users at once, all of them generating
        _stack('ruzinex_batch', 'ruzinex', 2048, 8, 240, 24, ragged=True),
        # a wide recurrent and attention hybrid answers one user
        _stack('tolenex_answer', 'tolenex', 4096, 1, 130, 24),
        # the smallest calls of the packed engine: a few tokens in, a few out
        _stack('narurax_small_call', 'narurax', 1024, 1, 5, 4),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng: random.Random):
    """A case of the same ranges: any design and weight form, from a handful of tokens to the longest prompts, one to eight requests."""
    while True:
        new = rng.choice([0, 0, _log_int(rng, 1, 24)])
        c = dict(batch=rng.choice([1, 1, 2, 3, 4, 5, 8]), prompt=_log_int(rng, 3, 4096), new=new, ragged=rng.random() < 0.5)
        if rng.random() < 0.4:
            c.update(path='llama', mode=rng.choice(['fp16', 'sq', 'woq8', 'woq4']), width=rng.choice([1024, 2048, 4096]),
                     layers=_log_int(rng, 4, 16), prompt=_log_int(rng, 3, 2000))  # positions up to 2048
        else:
            c.update(path=rng.choice(STACKS), width=rng.choice([512, 1024, 1536, 2048, 3072]), layers=4)
        if c['batch'] * c['prompt'] <= 4096:
            return c


def _lengths(case, rng):
    n = case['prompt']
    lens = [rng.randint(max(1, n // 2), n) if case['ragged'] else n for _ in range(case['batch'])]
    lens[0] = n
    return lens


def _prompts(case, seed):
    """[batch] lists of prompt + `new` token ids, and the prompts' lengths."""
    rng = random.Random(seed * 1000003 + 17)
    lens = _lengths(case, rng)
    ids = np.random.default_rng(seed).integers(3, VOCAB, (case['batch'], case['prompt'] + case['new']))
    return [ids[b, :lens[b] + case['new']].tolist() for b in range(case['batch'])], lens


# ------------------------------------------------------------------------------------------------------------------ weights
class _Rand(object):
    """Tensors drawn on the GPU in a fixed order from one generator."""

    def __init__(self, seed):
        self.g = torch.Generator(device='cuda').manual_seed(seed)

    def normal(self, *shape, s=1.0, mean=0.0):
        return torch.randn(shape, generator=self.g, device='cuda') * s + mean

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.g, device='cuda') * (hi - lo) + lo

    def integers(self, lo, hi, *shape, dtype):
        return torch.randint(lo, hi, shape, generator=self.g, device='cuda', dtype=dtype)


def _llama_ff(case):
    return int(case['width'] * 2.6875)


def _next_token(t):
    """What the random LLaMA models here answer: the head's row of next(t) is the embedding of t, so that the largest logit leads by a
    clear margin, as a trained model's does, and the answer does not hang on the last bit of a sum."""
    return (t * 7919 + 13) % VOCAB


def _llama_weights(case):
    """name -> tensor in the session's storage formats."""
    r, D, I, mode = _Rand(1), case['width'], _llama_ff(case), case['mode']
    t = {'vocab_embedding.weight': r.normal(VOCAB, D).half(), 'ln_f.weight': r.uniform(0.9, 1.1, D).half()}
    head = torch.empty_like(t['vocab_embedding.weight'])
    head[_next_token(torch.arange(VOCAB, device='cuda'))] = t['vocab_embedding.weight'] * D ** -0.5
    t['lm_head.weight'] = head

    def one(v):
        return torch.tensor([v], dtype=torch.float32, device='cuda')

    def linear(name, n, k):
        a = (6.0 / (n + k)) ** 0.5  # Xavier bound
        if mode == 'fp16':
            t[name + '.weight'] = r.uniform(-a, a, n, k).half()
        elif mode == 'sq':  # activations take about 28 steps per unit, rows of different scale
            t[name + '.weight'] = r.integers(-127, 128, n, k, dtype=torch.int8)
            t[name + '.per_channel_scale'] = (r.uniform(0.8, 1.2, 1, n) * (a / 127.0 / 28.0))
            t[name + '.act_scale'] = torch.ones((1, 1), dtype=torch.float32, device='cuda')
        else:
            bits = 8 if mode == 'woq8' else 4
            t[name + '.weight'] = r.integers(0, 256, n, k * bits // 8, dtype=torch.uint8)
            t[name + '.per_channel_scale'] = (r.uniform(0.8, 1.2, n) * (a / (127.0 if bits == 8 else 7.0))).half()

    for i in range(case['layers']):
        p = 'layers.%d.' % i
        t[p + 'input_layernorm.weight'] = r.uniform(0.9, 1.1, D).half()
        t[p + 'post_layernorm.weight'] = r.uniform(0.9, 1.1, D).half()
        linear(p + 'attention.qkv', 3 * D, D)
        linear(p + 'attention.dense', D, D)
        linear(p + 'mlp.fc', I, D)
        linear(p + 'mlp.gate', I, D)
        linear(p + 'mlp.proj', D, I)
        if mode == 'sq':
            t[p + 'input_layernorm.scale_to_int'] = one(28.0)
            t[p + 'post_layernorm.scale_to_int'] = one(28.0)
            t[p + 'attention.quantization_scaling_factor'] = one(60.0)
            t[p + 'mlp.quantization_scaling_factor'] = one(40.0)
        if mode != 'fp16':
            t[p + 'attention.kv_orig_quant_scale'] = one(127.0 / 6.0)
            t[p + 'attention.kv_quant_orig_scale'] = one(6.0 / 127.0)
    return t


def _expert_ff(width):
    return -(-int(width * 2.6875 / 4) // 64) * 64


def _stack_config(case):
    """config.json of a stack model with the layer sizes of a LLaMA-like model of this width (heads of 128, four query heads per key head)."""
    w, L, path = case['width'], case['layers'], case['path']
    heads, ff, eff = w // 128, int(w * 2.6875), _expert_ff(w)
    kv = max(heads // 4, 1)
    dense = {'kind': 'dense', 'ff': ff}
    if path == 'tolenex':  # every fourth layer an HGRN2 layer
        attn = {'type': 'attention', 'mlp': dense,
                'mixer': {'heads': heads, 'kv_heads': kv, 'dim': 64, 'vdim': 128, 'diff': 0.2, 'scale': 0.125, 'softcap': 30.0,
                          'rot': {'dims': 64, 'base': 500000.0, 'scaling': {'factor': 4.0, 'original': 8192, 'fast': 16.0, 'slow': 2.0}}}}
        rec = {'type': 'hgrn2', 'mlp': dense, 'mixer': {'heads': heads, 'dim': 128, 'vdim': 128}}
        return {'architecture': 'Tolenex', 'vocab': VOCAB, 'width': w, 'embedding': {'scale': 8.0}, 'norm': {'eps': 1e-6, 'groups': 4},
                'layers': [rec if i % 4 == 2 else attn for i in range(L)]}
    if path == 'rofozen':  # mamba2 / mamba2 / latent attention / mamba2 on the second layer's weights
        moe = {'kind': 'moe', 'expert': {'ff': eff},
               'router': {'experts': 32, 'identity': 2, 'top': 4, 'scale': 2.5, 'groups': {'count': 2, 'keep': 1}}}
        ssm = {'heads': 2 * w // 64, 'vdim': 64, 'state': 128, 'groups': 8, 'conv': 4, 'norm_groups': 8}
        lat = {'heads': heads, 'dim': 64, 'rot_dim': 64, 'vdim': 128, 'kv_rank': 256, 'q_rank': w * 3 // 8, 'scale': 128 ** -0.5,
               'mask': {'size': 512}, 'rot': {'dims': 64, 'base': 500000.0, 'scaling': {'factor': 4.0, 'original': 8192, 'fast': 32.0, 'slow': 1.0}}}
        layers = []
        for i in range(L):
            l = {'type': 'latent_attention' if i % 4 == 2 else 'mamba2', 'mixer': lat if i % 4 == 2 else ssm, 'mlp': moe if i else dense}
            layers.append(dict(l, weights_of=i - 2) if i % 4 == 3 else l)
        return {'architecture': 'Rofozen', 'vocab': VOCAB, 'width': w, 'norm': {'eps': 1e-6}, 'layers': layers}
    if path == 'narurax':  # attention_2 / channel_delta / attention / channel_delta
        moe = {'kind': 'moe', 'expert': {'ff': eff}, 'router': {'experts': 32, 'top': 4}}
        at = {'heads': heads, 'kv_heads': kv, 'dim': 128, 'vdim': 128, 'scale': 128 ** -0.5, 'mask': {'size': 512, 'keep_first': 4}}
        a2 = dict(at, rot={'dims': 128, 'base': 500000.0, 'scaling': {'factor': 8.0, 'low': 1.0, 'high': 4.0, 'original': 8192}})
        a1 = dict(at, rot={'dims': 64, 'base': 500000.0})
        dl = {'heads': heads, 'kv_heads': max(heads // 2, 1), 'dim': 128, 'vdim': 128, 'conv': 4}
        kinds = [('attention_2', a2), ('channel_delta', dl), ('attention', a1), ('channel_delta', dl)]
        return {'architecture': 'Narurax', 'vocab': VOCAB, 'width': w, 'norm': {'eps': 1e-6},
                'embedding': {'bigram': {'buckets': 65521, 'mul_prev': 1000003, 'mul_cur': 31}},
                'layers': [{'type': kinds[i % 4][0], 'mixer': kinds[i % 4][1], 'mlp': moe} for i in range(L)]}
    moe = {'kind': 'moe', 'expert': {'ff': eff}, 'router': {'experts': 32, 'top': 4}, 'shared': {'ff': 2 * eff}}

    def mixer(dim):
        return {'heads': heads, 'kv_heads': kv, 'dim': dim, 'vdim': 128, 'scale': dim ** -0.5, 'v_mix': True,
                'rot': {'dims': dim // 2, 'base': 500000.0, 'scaling': {'factor': 4.0}}}
    return {'architecture': 'Ruzinex', 'vocab': VOCAB, 'width': w, 'norm': {'eps': 1e-6}, 'residual_mult': 0.7,
            'layers': [{'type': 'attention', 'mixer': mixer(128 if i % 4 in (0, 3) else 192), 'mlp': moe if i % 2 else dense} for i in range(L)]}


def _stack_weights(case, cfg):
    """name -> bfloat16 tensor on the GPU, by the checkpoint's names."""
    r, t, W, path = _Rand(2), {}, case['width'], case['path']

    def put(name, a):
        t[name] = a.to(torch.bfloat16)

    def mat(name, *shape, s=1.0, mean=0.0):
        put(name, r.normal(*shape, s=s, mean=mean))

    def proj(name, n, k):
        mat(name, n, k, s=k ** -0.5)

    def norms(p, *names):
        for n in names:
            mat(p + n, W, s=0.1, mean=1.0)

    mat('embed', VOCAB, W, s=0.125 if path == 'tolenex' else 1.0)
    routers = [l['mlp']['router'] for l in cfg['layers'] if l['mlp']['kind'] == 'moe']
    if routers:
        # Which experts a token goes to is learned and mostly a matter of the token itself: its embedding holds four of these directions
        # (of one half of the experts, as the grouped choice wants it), and a layer's router reads them in an order of its own.  A router
        # of random rows would leave every twentieth choice to the last bit of a sum.
        ne = routers[0]['experts'] + routers[0].get('identity', 0)
        ways = torch.nn.functional.normalize(r.normal(ne, W), dim=1)
        mine = r.uniform(0, 1, VOCAB, ne // 2).argsort(1)[:, :4] + r.integers(0, 2, VOCAB, 1, dtype=torch.int64) * (ne // 2)
        t['embed'] = (t['embed'].float() + 12.0 * ways[mine].sum(1)).to(torch.bfloat16)
    if path == 'ruzinex':  # the embedding table is the head
        mat('final.norm', W, s=0.1 * W ** -0.5, mean=W ** -0.5)
    else:
        proj('head', VOCAB, W)
        norms('', 'final.norm')
    if path == 'narurax':
        mat('bigram', cfg['embedding']['bigram']['buckets'] + 1, W, s=0.5)
    for i, l in enumerate(cfg['layers']):
        if l.get('weights_of') is not None:
            continue
        p, m, mlp = 'l%d.' % i, l['mixer'], l['mlp']
        q, H, G, D, E = p + 'mix.', m['heads'], m.get('kv_heads'), m.get('dim'), m['vdim']
        norms(p, *(('norm1', 'norm1b', 'norm2', 'norm2b') if path == 'ruzinex' else ('norm1', 'norm2')))
        if path == 'tolenex':
            for n in ('1', '2'):
                proj(p + 'rg' + n, W, W)
                mat(p + 'rg' + n + '.b', W, s=0.5)
        if path == 'narurax':
            put(p + 'shift', r.uniform(0.0, 1.0, W))
        if l['type'] == 'hgrn2':
            proj(q + 'q', H * D, W), proj(q + 'f', H * D, W), proj(q + 'v', H * E, W)
            mat(q + 'f.b', H * D, mean=1.0)
            put(q + 'lower', r.uniform(0.0, 0.9, H * D))
            mat(q + 'norm', E, s=0.1, mean=1.0)
        elif l['type'] == 'mamba2':
            N, K, inner = m['state'], m['conv'], H * E
            ch = inner + 2 * m['groups'] * N
            proj(q + 'in', inner + ch + H, W)
            mat(q + 'conv', ch, K, s=K ** -0.5), mat(q + 'conv.b', ch, s=0.1), mat(q + 'dt_bias', H, s=0.5, mean=-1.0)
            put(q + 'A_log', r.uniform(0.5, 4.0, H).log())
            mat(q + 'D', H, s=0.3, mean=1.0), mat(q + 'norm', inner, s=0.1, mean=1.0)
        elif l['type'] == 'latent_attention':
            C, Q, R = m['kv_rank'], m['q_rank'], m['rot_dim']
            proj(q + 'dq', Q, W), mat(q + 'dq.norm', Q, s=0.1, mean=1.0), proj(q + 'uq', H * (D + R), Q)
            proj(q + 'dkv', C + R, W), mat(q + 'dkv.norm', C, s=0.1, mean=1.0), proj(q + 'uk', H * D, C), proj(q + 'uv', H * E, C)
            mat(q + 'sink', H, s=0.5)
        elif l['type'] == 'channel_delta':
            rank = max(8, W // 16)
            for n, rows in (('q', G * D), ('k', G * D), ('v', H * E)):
                proj(q + n, rows, W), mat(q + n + '.conv', rows, m['conv'], s=m['conv'] ** -0.5)
            proj(q + 'b', H, W)
            put(q + 'A_log', r.uniform(0.05, 1.0, H).log())
            mat(q + 'norm', E, s=0.1, mean=1.0), mat(q + 'dt_bias', H * D, s=0.5, mean=-1.0)
            proj(q + 'a1', rank, W), proj(q + 'a2', H * D, rank), proj(q + 'g1', rank, W), proj(q + 'g2', H * E, rank)
        elif path == 'tolenex':
            proj(q + 'q', H * 2 * D, W), proj(q + 'k', G * 2 * D, W), proj(q + 'v', G * E, W)
            for n in ('lq1', 'lk1', 'lq2', 'lk2'):
                mat(q + n, D, s=0.3)
        else:
            proj(q + 'q', H * D, W), proj(q + 'k', G * D, W)
            if path == 'narurax' and l['type'] == 'attention':
                put(q + 'talk', torch.eye(H, device='cuda') + r.normal(H, H, s=0.3 * H ** -0.5))
                proj(q + 'g', H * E, W)
            else:
                proj(q + 'v', G * E, W)
                mat(q + 'q.b', H * D, s=0.1), mat(q + 'k.b', G * D, s=0.1), mat(q + 'v.b', G * E, s=0.1)
            if l['type'] == 'attention_2':
                mat(q + 'o.b', W, s=0.1), mat(q + 'q.norm', D, s=0.1, mean=1.0), mat(q + 'k.norm', D, s=0.1, mean=1.0)
            else:
                mat(q + 'sink', H, s=0.5)
            if path == 'ruzinex':
                put(q + 'vmix', r.normal(s=0.1, mean=0.5))
        proj(q + 'o', W, H * E)
        p += 'mlp.'
        parts = [('', mlp['ff'])] if mlp['kind'] == 'dense' else [('e%d.' % e, mlp['expert']['ff']) for e in range(mlp['router']['experts'])]
        if mlp['kind'] == 'moe':
            half = r.uniform(0, 1, 2, ne // 2).argsort(1) + torch.tensor([[0], [ne // 2]], device='cuda')
            put(p + 'router', 0.5 * ways[half.flatten()])
            if path == 'rofozen':
                mat(p + 'correction', ne, s=0.5 / ne)
            if path == 'ruzinex':
                mat(p + 'router.b', ne, s=0.1), proj(p + 'shared.sg', 1, W)
                parts.append(('shared.', mlp['shared']['ff']))
        for n, F in parts:
            proj(p + n + 'gate', F, W), proj(p + n + 'up', F, W), proj(p + n + 'down', W, F)
    return t


# ------------------------------------------------------------------------------------------------------------------ the engines
_held = {}  # the engine that the program keeps: the last one that was asked for


def _held_engine(key, make):
    if key not in _held:
        for old in _held.values():
            getattr(old, 'engine', old).close()
        _held.clear()
        gc.collect()
        torch.cuda.empty_cache()
        _held[key] = make()
    return _held[key]


def _llama_session(case):
    from tensorrt_llm.runtime.native import NativeSession
    D = case['width']
    s = NativeSession(dict(num_layers=case['layers'], num_heads=D // 128, hidden_size=D, inter_size=_llama_ff(case), vocab_size=VOCAB,
                           max_position_embeddings=2048, rms_norm_eps=1e-6, quant_mode=QUANT_MODE[case['mode']]))
    for name, t in _llama_weights(case).items():
        s.set_tensor(name, t)
    torch.cuda.synchronize()
    s.finalize()
    s.setup(case['batch'], case['prompt'], case['new'])
    return s


def _stack_session(case):
    from tensorrt_llm import models
    from tensorrt_llm.runtime import RaggedGenerationSession
    cfg = _stack_config(case)
    tensors = {n: (t.view(torch.int16).cpu().numpy().view(np.uint16), 'bfloat16') for n, t in _stack_weights(case, cfg).items()}
    cls = getattr(models, cfg['architecture'] + 'ForCausalLM')
    model = cls(cls.config_class(cfg), tensors)
    pages = -(-(case['prompt'] + case['new']) // model.page_size)
    return RaggedGenerationSession(model, dtype='bfloat16', max_tokens=case['batch'] * pages * model.page_size, max_sequences=case['batch'],
                                   max_batch_tokens=BUDGET)


def prepare(case, seed):
    tokens, lens = _prompts(case, seed)
    key = tuple(sorted((k, v) for k, v in case.items() if k not in ('name', 'ragged')))
    if case['path'] == 'llama':
        s = _held_engine(key, lambda: _llama_session(case))
        ids = np.full((case['batch'], case['prompt']), 2, np.int32)
        for b, n in enumerate(lens):
            ids[b, :n] = tokens[b][:n]
        return dict(session=s, ids=ids, lens=np.asarray(lens, np.int32), new=case['new'])
    s = _held_engine(key, lambda: _stack_session(case))
    return dict(session=s, steps=_steps(tokens, lens, case['new']), last=list(range(case['batch'])))


def _steps(tokens, lens, new):
    """The steps of a batch of requests: [(request, tokens, wanted places)] each.  Prompts first, cut where a step's budget ends, then
    one token of every request per step."""
    steps, step, room = [], [], BUDGET
    for b, n in enumerate(lens):
        fed = 0
        while fed < n:
            take = min(room, n - fed)
            want = [] if fed + take < n else [take - 1] if new else list(range(max(0, take - 4), take))
            step.append((b, tokens[b][fed:fed + take], want))
            fed, room = fed + take, room - take
            if not room:
                steps.append(step)
                step, room = [], BUDGET
    if step:
        steps.append(step)
    return steps + [[(b, [tokens[b][n + i]], [0]) for b, n in enumerate(lens)] for i in range(new)]


def run(state):
    s = state['session']
    if 'ids' in state:
        if not state['new']:
            s.context(state['ids'], state['lens'])
            return {'logits': s.logits()}
        ids = s.generate(state['ids'], state['lens'], state['new'])
        return {'tokens': ids, 'logits': s.logits()}
    out = []
    for i, step in enumerate(state['steps']):
        logits, _ = s.step(step, end=state['last'] if i == len(state['steps']) - 1 else ())
        if logits is not None:
            out.append(logits)
    return out


# ------------------------------------------------------------------------------------------------------------------ bytes, operations, tolerances
def _mean_lengths(case):
    return [float(case['prompt'])] + [0.75 * case['prompt'] if case['ragged'] else float(case['prompt'])] * (case['batch'] - 1)


def work(case):
    """Weights are read once per step that needs them (a step's tokens hang on the step before), caches once per generated token;
    routed layers read the experts that this many tokens are expected to reach."""
    lens, new, D = _mean_lengths(case), case['new'], case['width']
    rows, gen = sum(lens), max(new - 1, 0) if case['path'] == 'llama' else new
    steps = [(rows, 1.0)] + ([(float(case['batch']), float(gen))] if gen else [])  # (rows of a step, steps like it)
    if case['path'] != 'llama' and rows > BUDGET:
        steps[0] = (rows / math.ceil(rows / BUDGET), float(math.ceil(rows / BUDGET)))
    if case['path'] == 'llama':
        I, esz = _llama_ff(case), {'fp16': 2.0, 'sq': 1.0, 'woq8': 1.0, 'woq4': 0.5}[case['mode']]
        per_layer = 4 * D * D + 3 * D * I
        kv = 2 * D * (2 if case['mode'] == 'fp16' else 1)
        nbytes = sum(k * (case['layers'] * per_layer * esz + VOCAB * D * 2 + case['batch'] * VOCAB * 4) for _, k in steps)
        nbytes += case['layers'] * kv * sum(n + gen * (n + gen / 2) for n in lens)
        flops = case['layers'] * (2.0 * per_layer * (rows + gen * case['batch']) + sum(2 * D * (n * n + 2 * gen * (n + gen / 2)) for n in lens))
        return {'bytes': nbytes, 'flops': flops + 2.0 * VOCAB * D * case['batch'] * (1 + gen)}
    cfg, nbytes, flops = _stack_config(case), 0.0, 0.0
    wanted = len(lens) * (1 if new else 4)
    for r, k in steps:
        nbytes += k * (VOCAB * D * 2 + (wanted if r == steps[0][0] else len(lens)) * VOCAB * 4)
    flops += 2.0 * VOCAB * D * (wanted + gen * len(lens))
    for l in cfg['layers']:
        m, mlp = l['mixer'], l['mlp']
        H, E, dim, G = m['heads'], m['vdim'], m.get('dim', 0), m.get('kv_heads', m['heads'])
        span, cache, score, state = (m.get('mask') or {}).get('size', 1 << 30), 0, 0, 0
        w = D * H * E  # the output projection
        if l['type'] == 'mamba2':
            w += D * (2 * H * E + 2 * m['groups'] * m['state'] + H)
            state = H * E * m['state']
        elif l['type'] == 'hgrn2':
            w += D * (2 * H * dim + H * E)
            state = H * E * dim
        elif l['type'] == 'channel_delta':
            w += D * (2 * G * dim + H * E + H + D // 8) + (D // 16) * H * (dim + E)
            state = H * E * dim
        elif l['type'] == 'latent_attention':
            w += D * (m['q_rank'] + m['kv_rank'] + m['rot_dim']) + m['q_rank'] * H * (dim + m['rot_dim']) + m['kv_rank'] * H * (dim + E)
            cache, score = m['kv_rank'] + m['rot_dim'], H * (dim + m['rot_dim'] + E)
        else:
            maps = 2 if case['path'] == 'tolenex' else 1
            own = 0 if case['path'] == 'narurax' and l['type'] == 'attention' else E  # that mixer's values are its keys
            w += D * (maps * H * dim + maps * G * dim + G * own) + (0 if own else D * H * E)
            cache, score = G * (maps * dim + own), H * maps * (dim + E)
        if case['path'] == 'tolenex':
            w += 2 * D * D
        for r, k in steps:
            nbytes += k * (2 * w + (8 * state * len(lens) if state else 0))
            flops += k * r * (2.0 * w + 6.0 * state)
            one = 3 * D * (mlp['ff'] if mlp['kind'] == 'dense' else mlp['expert']['ff'])
            if mlp['kind'] == 'dense':
                nbytes, flops = nbytes + k * 2 * one, flops + k * r * 2.0 * one
                continue
            e, top = mlp['router']['experts'], mlp['router']['top']
            sh = 3 * D * (mlp.get('shared') or {}).get('ff', 0)
            nbytes += k * 2 * (one * e * (1 - (1 - top / e) ** r) + sh + D * e)
            flops += k * r * 2.0 * (one * top + sh + D * e)
        for n in lens:
            seen = n * (n + 1) / 2 if n <= span else span * (span + 1) / 2 + (n - span) * span
            nbytes += 2 * cache * (n + gen * min(n + gen / 2, span))
            flops += 2.0 * score * (seen + gen * min(n + gen / 2, span))
    return {'bytes': nbytes, 'flops': flops}


def tolerance(case):
    """About four times what the results are off their 64-bit values: fp16 and weight-only LLaMA 1e-3 to 4e-3; SmoothQuant 3e-2 (a quantiser
    that rounds the other way moves its row by a whole step, 256 of them in a row of layers); bfloat16 stacks 3e-3 to 1e-2."""
    return {'rel': {'sq': 8e-2, 'fp16': 1e-2, 'woq8': 1.5e-2, 'woq4': 1.5e-2}.get(case.get('mode'), 3e-2), 'differ': 0.0}


# ------------------------------------------------------------------------------------------------------------------ 64-bit results
def _rms(x, w, eps=1e-6):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _turn(x, ang, mult, halves):
    """x [n, heads, d]: the first 2 * ang.shape[1] dimensions turn, in pairs of neighbours or of halves."""
    k = ang.shape[1]
    c, s = (torch.cos(ang) * mult)[:, None], (torch.sin(ang) * mult)[:, None]
    u, v = (x[..., :k], x[..., k:2 * k]) if halves else (x[..., 0:2 * k:2], x[..., 1:2 * k:2])
    a, b = u * c - v * s, v * c + u * s
    turned = torch.cat([a, b], -1) if halves else torch.stack([a, b], -1).flatten(-2)
    return torch.cat([turned, x[..., 2 * k:]], -1)


def _angles(n, rot):
    """(position x frequency [n, dims / 2], multiplier of cos and sin)."""
    d, base, sc, mult = rot['dims'], rot['base'], rot.get('scaling'), 1.0
    i = torch.arange(d // 2, dtype=torch.float64, device='cuda')
    f = base ** (-2.0 * i / d)
    if sc and 'fast' in sc:  # YaRN
        lo, hi = [d * math.log(sc['original'] / (2 * math.pi * sc[t])) / (2 * math.log(base)) for t in ('fast', 'slow')]
        lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), d - 1)
        ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        f, mult = f / sc['factor'] * ramp + f * (1 - ramp), 0.1 * math.log(sc['factor']) + 1.0
    elif sc and 'low' in sc:  # three bands by wavelength
        turns = sc['original'] * f / (2 * math.pi)
        s = ((turns - sc['low']) / (sc['high'] - sc['low'])).clamp(0, 1)
        f = (1 - s) * f / sc['factor'] + s * f
    elif sc:
        f = f / sc['factor']
    return torch.arange(n, dtype=torch.float64, device='cuda')[:, None] * f, mult


def _attend(q, k, v, vis, scale, cap=0.0, sink=None, mix=None):
    """q [n, H, d], k [n, G, d], v [n, G, e] -> [n, H, e]."""
    H, per = q.shape[1], q.shape[1] // k.shape[1]
    s = torch.matmul(q.transpose(0, 1), k.repeat_interleave(per, 1).permute(1, 2, 0)) * scale
    if cap:
        s = cap * torch.tanh(s / cap)
    s = s.masked_fill(~vis, -math.inf)
    top = s.amax(-1, keepdim=True)
    if sink is not None:
        top = torch.maximum(top, sink.view(H, 1, 1))
    s = torch.exp(s - top)
    den = s.sum(-1, keepdim=True)
    if sink is not None:
        den = den + torch.exp(sink.view(H, 1, 1) - top)
    s = s / den
    if mix is not None:
        s = (mix @ s.flatten(1)).view_as(s)
    return torch.matmul(s, v.repeat_interleave(per, 1).transpose(0, 1)).transpose(0, 1)


def _visible(n, mask):
    i = torch.arange(n, device='cuda')
    d = i[:, None] - i
    vis = d >= 0
    return vis & ((d < mask['size']) | (i < mask.get('keep_first', 0))[None]) if mask else vis


def _conv(u, kernel, bias=None):
    n, taps = u.shape[0], kernel.shape[1]
    u = torch.cat([u.new_zeros(taps - 1, u.shape[1]), u])
    y = sum(u[k:k + n] * kernel[:, k] for k in range(taps))
    return torch.nn.functional.silu(y if bias is None else y + bias)


def _scan(decay, key, value, query):
    """S <- decay * S + key value^T, out = S^T query: decay, key, query [n, H, d], value [n, H, e]."""
    S, out = key.new_zeros(key.shape[1], key.shape[2], value.shape[2]), torch.empty_like(value)
    for t in range(key.shape[0]):
        S.mul_(decay[t, :, :, None]).addcmul_(key[t, :, :, None], value[t, :, None, :])
        torch.bmm(query[t, :, None], S, out=out[t, :, None])
    return out


def _delta_scan(q, k, v, beta, g):
    S, out = k.new_zeros(k.shape[1], k.shape[2], v.shape[2]), torch.empty_like(v)
    for t in range(k.shape[0]):
        S.mul_(g[t, :, :, None])
        u = beta[t, :, None] * (v[t] - torch.bmm(k[t, :, None], S)[:, 0])
        S.addcmul_(k[t, :, :, None], u[:, None, :])
        torch.bmm(q[t, :, None], S, out=out[t, :, None])
    return out


class _StackReference(object):
    """One sequence through a stack model in 64 bits."""

    def __init__(self, case):
        self.path, self.cfg = case['path'], _stack_config(case)
        self.t = _stack_weights(case, self.cfg)

    def w(self, name):
        return self.t[name].double()

    def mul(self, x, name):
        return x @ self.w(name).T

    def mixer(self, l, q, h):
        m, n, w, mul = l['mixer'], h.shape[0], self.w, self.mul
        H, G, D, E = m['heads'], m.get('kv_heads'), m.get('dim'), m['vdim']
        ang, mult = _angles(n, m['rot']) if 'rot' in m else (None, 1.0)
        vis = _visible(n, m.get('mask'))
        if l['type'] == 'hgrn2':
            f = w(q + 'lower') + (1 - w(q + 'lower')) * torch.sigmoid(mul(h, q + 'f') + w(q + 'f.b'))
            f = f.view(n, H, D)
            o = _scan(f, 1 - f, mul(h, q + 'v').view(n, H, E), torch.nn.functional.silu(mul(h, q + 'q')).view(n, H, D))
            return mul(_rms(o, w(q + 'norm')).flatten(1), q + 'o')
        if l['type'] == 'mamba2':
            inner, N, g = H * E, m['state'], m['groups']
            z, xbc, dt = mul(h, q + 'in').split([inner, inner + 2 * g * N, H], 1)
            x, b, c = _conv(xbc, w(q + 'conv'), w(q + 'conv.b')).split([inner, g * N, g * N], 1)
            x, b, c = x.view(n, H, E), [v.view(n, g, N).repeat_interleave(H // g, 1) for v in (b, c)][0], c.view(n, g, N).repeat_interleave(H // g, 1)
            dt = torch.nn.functional.softplus(dt + w(q + 'dt_bias'), threshold=1e9)[:, :, None]
            y = _scan(torch.exp(-w(q + 'A_log').exp()[:, None] * dt), dt * b, x, c) + w(q + 'D')[:, None] * x
            y = (y.flatten(1) * torch.nn.functional.silu(z)).view(n, m['norm_groups'], -1)
            return mul(_rms(y, 1.0).flatten(1) * w(q + 'norm'), q + 'o')
        if l['type'] == 'latent_attention':
            C = m['kv_rank']
            a = mul(_rms(mul(h, q + 'dq'), w(q + 'dq.norm')), q + 'uq').view(n, H, -1)
            kv = mul(h, q + 'dkv')
            c = _rms(kv[:, :C], w(q + 'dkv.norm'))
            kr = _turn(kv[:, None, C:], ang, mult, True).expand(n, H, -1)
            a = torch.cat([a[..., :D], _turn(a[..., D:], ang, mult, True)], -1)
            k = torch.cat([mul(c, q + 'uk').view(n, H, D), kr], -1)
            return mul(_attend(a, k, mul(c, q + 'uv').view(n, H, E), vis, m['scale'], sink=w(q + 'sink')).flatten(1), q + 'o')
        if l['type'] == 'channel_delta':
            a, k, v = [_conv(mul(h, q + s), w(q + s + '.conv')).view(n, c, -1) for s, c in (('q', G), ('k', G), ('v', H))]
            a, k = [(x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 1) for x in (a, k)]
            step = torch.nn.functional.softplus(mul(mul(h, q + 'a1'), q + 'a2') + w(q + 'dt_bias'), threshold=1e9).view(n, H, D)
            o = _delta_scan(a * D ** -0.5, k, v, torch.sigmoid(mul(h, q + 'b')), torch.exp(-w(q + 'A_log').exp()[:, None] * step))
            return mul(_rms(o, w(q + 'norm')).flatten(1) * torch.sigmoid(mul(mul(h, q + 'g1'), q + 'g2')), q + 'o')
        if self.path == 'tolenex':
            a, k, v = mul(h, q + 'q').view(n, 2 * H, D), mul(h, q + 'k').view(n, 2 * G, D), mul(h, q + 'v').view(n, G, E)
            a, k = [_turn(x, ang, mult, False).view(n, -1, 2, D) for x in (a, k)]
            lam = (w(q + 'lq1') * w(q + 'lk1')).sum().exp() - (w(q + 'lq2') * w(q + 'lk2')).sum().exp() + m['diff']
            o = [_attend(a[:, :, i], k[:, :, i], v, vis, m['scale'], m['softcap']) for i in range(2)]
            return mul((_rms(o[0] - lam * o[1], 1.0) * (1 - m['diff'])).flatten(1), q + 'o')
        if self.path == 'ruzinex':
            a, k, v = [(mul(h, q + s) + w(q + s + '.b')).view(n, c, -1) for s, c in (('q', H), ('k', G), ('v', G))]
            if self.first is None:
                self.first = v
            else:
                v = (1 - w(q + 'vmix')) * v + w(q + 'vmix') * self.first
            a, k = _turn(a, ang, mult, True), _turn(k, ang, mult, True)
            return mul(_attend(a, k, v, vis, m['scale'], sink=w(q + 'sink')).flatten(1), q + 'o')
        if l['type'] == 'attention_2':
            a, k, v = [(mul(h, q + s) + w(q + s + '.b')).view(n, c, -1) for s, c in (('q', H), ('k', G), ('v', G))]
            a, k = _turn(_rms(a, w(q + 'q.norm')), ang, mult, False), _turn(_rms(k, w(q + 'k.norm')), ang, mult, False)
            return mul(_attend(a, k, v, vis, m['scale'], sink=a.new_zeros(H)).flatten(1), q + 'o') + w(q + 'o.b')
        a, k = mul(h, q + 'q').view(n, H, D), mul(h, q + 'k').view(n, G, D)
        o = _attend(_turn(a, ang, mult, False), _turn(k, ang, mult, False), k, vis, m['scale'], sink=w(q + 'sink'), mix=w(q + 'talk'))
        return mul(o.flatten(1) * torch.sigmoid(mul(h, q + 'g')), q + 'o')

    def gated(self, x, p, act):
        return self.mul(act(self.mul(x, p + 'gate')) * self.mul(x, p + 'up'), p + 'down')

    def feed_forward(self, mlp, p, h):
        F = torch.nn.functional
        if mlp['kind'] == 'dense':
            return self.gated(h, p, lambda x: F.gelu(x, approximate='tanh'))
        r, z = mlp['router'], self.mul(h, p + 'router')
        y = torch.zeros_like(h)
        if self.path == 'rofozen':
            s = torch.softmax(z, -1)
            choice, g = s + self.w(p + 'correction'), r['groups']
            best = choice.view(len(h), g['count'], -1).amax(-1).topk(g['keep'], -1).indices
            kept = torch.zeros(len(h), g['count'], dtype=torch.bool, device='cuda').scatter_(1, best, True)
            chosen = choice.masked_fill(~kept.repeat_interleave(z.shape[1] // g['count'], 1), -math.inf).topk(r['top'], -1).indices
            weight = s.gather(1, chosen) * r['scale']
            y = y + (weight * (chosen >= r['experts'])).sum(1, keepdim=True) * h
        elif self.path == 'ruzinex':
            top = (z + self.w(p + 'router.b')).topk(r['top'], -1)
            chosen, weight = top.indices, torch.softmax(top.values, -1)
            y = y + torch.sigmoid(self.mul(h, p + 'shared.sg')) * self.gated(h, p + 'shared.', F.silu)
        else:
            chosen = z.topk(r['top'], -1).indices
            weight = torch.sigmoid(z).gather(1, chosen)
        for e in range(r['experts']):
            rows, place = (chosen == e).nonzero(as_tuple=True)
            if len(rows):
                g = weight[rows, place][:, None]
                a = self.gated(h[rows] * g if self.path == 'narurax' else h[rows], p + 'e%d.' % e, F.silu)
                y.index_add_(0, rows, a if self.path == 'narurax' else a * g)
        return y

    def logits(self, tokens, places):
        cfg, w, path = self.cfg, self.w, self.path
        ids, groups = torch.tensor(tokens, device='cuda'), 4 if path == 'tolenex' else 1

        def norm(x, name):
            return _rms(x.view(len(x), groups, -1), 1.0).view_as(x) * w(name)

        x, self.first = self.t['embed'][ids].double(), None
        if path == 'tolenex':
            x = x * cfg['embedding']['scale']
        if path == 'narurax':
            b = cfg['embedding']['bigram']
            rows = torch.cat([ids.new_tensor([b['buckets']]), (ids[:-1] * b['mul_prev'] + ids[1:] * b['mul_cur']) % b['buckets']])
            x = x + self.t['bigram'][rows].double()
        for i, l in enumerate(cfg['layers']):
            p = 'l%d.' % l.get('weights_of', i)
            h = norm(x, p + 'norm1')
            if path == 'narurax':
                h = h + (torch.cat([h.new_zeros(1, h.shape[1]), h[:-1]]) - h) * w(p + 'shift')
            y = self.mixer(l, p + 'mix.', h)
            if path == 'tolenex':
                h2 = norm(x, p + 'norm2')
                x = x + y * torch.sigmoid(self.mul(h, p + 'rg1') + w(p + 'rg1.b'))
                x = x + self.feed_forward(l['mlp'], p + 'mlp.', h2) * torch.sigmoid(self.mul(h2, p + 'rg2') + w(p + 'rg2.b'))
            elif path == 'ruzinex':
                x = x + cfg['residual_mult'] * norm(y, p + 'norm1b')
                x = x + cfg['residual_mult'] * norm(self.feed_forward(l['mlp'], p + 'mlp.', norm(x, p + 'norm2')), p + 'norm2b')
            else:
                x = x + y
                x = x + self.feed_forward(l['mlp'], p + 'mlp.', norm(x, p + 'norm2'))
        return self.mul(norm(x[places], 'final.norm'), 'embed' if path == 'ruzinex' else 'head')


def _stack_exact(case, seed):
    tokens, lens = _prompts(case, seed)
    ref = _StackReference(case)
    rows = {}
    for b, n in enumerate(lens):
        places = list(range(n - 1, n + case['new'])) if case['new'] else list(range(max(0, n - 4), n))
        for place, row in zip(places, ref.logits(tokens[b], places)):
            rows[b, place] = row
    out, at = [], [0] * case['batch']
    for step in _steps(tokens, lens, case['new']):
        got = [rows[b, at[b] + p] for b, _, want in step for p in want]
        for b, toks, _ in step:
            at[b] += len(toks)
        if got:
            out.append(torch.stack(got))
    return out


def _llama_exact(case, seed):
    tokens, lens = _prompts(case, seed)
    t, D, mode, new = _llama_weights(case), case['width'], case['mode'], case['new']
    H = D // 128
    seqs = []
    for b, n in enumerate(lens):  # the answer is known ahead, token by token; the largest logits below confirm it
        s = tokens[b][:n]
        for _ in range(max(new - 1, 0)):
            s.append(_next_token(s[-1]))
        seqs.append(s)
    ends = np.cumsum([len(s) for s in seqs]).tolist()
    spans = list(zip([0] + ends, ends, lens))
    place = torch.arange(128 // 2, dtype=torch.float64, device='cuda')
    freq = 10000.0 ** (-place / 64)

    def linear(x, name, scale=None):
        w = t[name + '.weight']
        if mode == 'fp16':
            return x @ w.double().T
        if mode == 'sq':
            q = (x * scale.double()).round().clamp(-128, 127)
            return q @ w.double().T * t[name + '.per_channel_scale'].double()
        if mode == 'woq8':
            return x @ (w.double() - 128).T * t[name + '.per_channel_scale'].double()
        v = torch.stack([w & 15, w >> 4], -1).view(w.shape[0], -1, 8)  # a word's nibbles hold elements 0 2 4 6 1 3 5 7
        v = v[..., [0, 4, 1, 5, 2, 6, 3, 7]].flatten(1)
        return x @ (v.double() - 8).T * t[name + '.per_channel_scale'].double()

    def cached(x, p):
        if mode == 'fp16':
            return x
        s = [t[p + 'attention.kv_%s_scale' % n].double() for n in ('orig_quant', 'quant_orig')]
        return (x * s[0]).round().clamp(-128, 127) * s[1]

    x = t['vocab_embedding.weight'][torch.tensor(sum(seqs, []), device='cuda')].double()
    for i in range(case['layers']):
        p = 'layers.%d.' % i
        scales = [t.get(p + n) for n in ('input_layernorm.scale_to_int', 'attention.quantization_scaling_factor',
                                         'post_layernorm.scale_to_int', 'mlp.quantization_scaling_factor')]
        qkv = linear(_rms(x, t[p + 'input_layernorm.weight'].double()), p + 'attention.qkv', scales[0]).view(-1, 3, H, 128)
        ctx = torch.empty_like(qkv[:, 0])
        for lo, hi, n in spans:
            ang = torch.arange(hi - lo, dtype=torch.float64, device='cuda')[:, None] * freq
            q, k, v = _turn(qkv[lo:hi, 0], ang, 1.0, True), _turn(qkv[lo:hi, 1], ang, 1.0, True), qkv[lo:hi, 2]
            vis = _visible(hi - lo, None)
            ctx[lo:lo + n] = _attend(q[:n], k[:n], v[:n], vis[:n, :n], 128 ** -0.5)
            for a in range(n, hi - lo):  # a generated token reads the cache, and its own key and value as they are
                kc, vc = torch.cat([cached(k[:a], p), k[a:a + 1]]), torch.cat([cached(v[:a], p), v[a:a + 1]])
                ctx[lo + a] = _attend(q[a:a + 1], kc, vc, vis[a:a + 1, :a + 1], 128 ** -0.5)[0]
        x = x + linear(ctx.flatten(1), p + 'attention.dense', scales[1])
        h = _rms(x, t[p + 'post_layernorm.weight'].double())
        a = torch.nn.functional.silu(linear(h, p + 'mlp.fc', scales[2])) * linear(h, p + 'mlp.gate', scales[2])
        x = x + linear(a, p + 'mlp.proj', scales[3])
    logits = _rms(x, t['ln_f.weight'].double()) @ t['lm_head.weight'].double().T
    last = torch.stack([logits[hi - 1] for _, hi, _ in spans])
    if not new:
        return {'logits': last}
    out = np.full((case['batch'], case['prompt'] + new), 2, np.int32)
    for b, (lo, hi, n) in enumerate(spans):
        out[b, :n] = tokens[b][:n]
        out[b, case['prompt']:] = logits[lo + n - 1:hi].argmax(-1).cpu().numpy()
    return {'tokens': out, 'logits': last}


def exact(case, seed):
    return _llama_exact(case, seed) if case['path'] == 'llama' else _stack_exact(case, seed)
