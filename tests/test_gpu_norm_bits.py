"""Norms to the last bit: the fp32 sum of squares in the order that its launch has (a lane's four squares, a tree over 64 lanes, the waves in turn), which the order of the
compiler's own contractions would otherwise change with the code around it.  A value of a normed bfloat16 row turns over one time in 30000 where its row's sum is another in
the last bit: rows enough that this shows, which each test asks of its inputs first."""
import numpy as np
import pytest

import narurax_cases as N
import rofozen_cases as F
import test_gpu_narurax
import test_gpu_rofozen
import test_gpu_tolenex
import tolenex_cases as T
from tolenex_cases import bf16_round

pytestmark = pytest.mark.gpu
f32 = np.float32


def fma(a, b, c):
    return (a.astype(np.longdouble) * b + c).astype(f32)


def sum_squares(x, x_first):
    """Rows of `threads` lanes with one float4 of every 4096 values each."""
    n, width = x.shape
    threads = min(1024, -(-width // 256) * 64)
    x = np.concatenate([x, np.zeros((n, -width % (4 * threads)), f32)], 1).reshape(n, -1, threads, 4)
    a, b = (x[..., 0], x[..., 1]) if x_first else (x[..., 1], x[..., 0])
    s = fma(b, b, a * a)
    for k in (2, 3):
        s = fma(x[..., k], x[..., k], s)
    lanes = s[:, 0]
    for k in range(1, s.shape[1]):
        lanes = lanes + s[:, k]
    tree = lanes.reshape(n, -1, 64)
    while tree.shape[2] > 1:
        tree = tree[..., ::2] + tree[..., 1::2]
    total = np.zeros(n, f32)
    for wave in tree[..., 0].T:
        total = total + wave
    return total


def normed(x, w, total, eps):
    return bf16_round(x * (f32(1) / np.sqrt(total / f32(x.shape[1]) + f32(eps)))[:, None] * w)


def embedded(cfg, w, toks):
    b = cfg['embedding']['bigram']
    return w['embed'][toks] + w['bigram'][[b['buckets']] + [(i * b['mul_prev'] + j * b['mul_cur']) % b['buckets'] for i, j in zip(toks, toks[1:])]]


def one_stream(width):
    """A layer that adds nothing, rows with bits down to 2^-24 of themselves, most of a row's sum in two squares, columns one by one by a head that is the identity."""
    cfg = N.make_config([N.attn_layer(heads=2, kv_heads=1)], width=width, vocab=width)
    w = N.random_weights(cfg, 5)
    w['l0.mix.o'][:] = 0
    w['bigram'] = bf16_round(w['bigram'] / 300)
    w['embed'][:, 8:10] *= 128
    w['bigram'][:, 8:10] *= 128
    w['head'] = np.eye(width, dtype=f32)
    return cfg, w, np.random.default_rng(3).permutation(width)[:2000].tolist()


@pytest.mark.parametrize('width', [1000, 2048, 4104])
def test_norm_of_one_stream(width):
    cfg, w, toks = one_stream(width)
    x = embedded(cfg, w, toks)
    want, other = (normed(x, w['final.norm'], sum_squares(x, first), cfg['norm']['eps']) for first in (True, False))
    assert (want != other).any()
    s = test_gpu_narurax.session_for(cfg, w, 'bfloat16', max_tokens=2048, max_sequences=1)
    np.testing.assert_array_equal(s.step([('a', toks, list(range(len(toks))))])[0], want)


def small(**kw):
    return dict(heads=2, vdim=16, state=16, groups=1, norm_groups=1, **kw)


LONE = {
    **{f'one stream of {width}': (F, F.make_config([F.mamba_layer(**small(mlp=F.dense(ff=40))), F.latent_layer(mlp=F.moe(experts=4, identity=2, top=2, count=1, keep=1)),
                                                    F.mamba_layer(**small(mlp=None)), F.mamba_layer(**small(mlp=F.dense(ff=24)))], width=width)) for width in (96, 1024, 1040, 2048, 3088, 4096)},
    'one stream of 4096 and many columns': (F, F.make_config([F.mamba_layer(heads=70, vdim=32, state=8, groups=1, norm_groups=1, mlp=F.dense(ff=40))] * 2, width=4096)),
    **{f'{groups} parts of {width}': (T, T.make_config([T.attention_layer(heads=2, kv_heads=1, dim=16, vdim=16, rot_dims=8, ff=40), T.hgrn2_layer(heads=2, dim=16, vdim=16, ff=24)],
                                                       width=width, groups=groups)) for width, groups in ((96, 1), (96, 2), (1040, 4), (2048, 1), (2064, 2), (2048, 8), (4096, 1), (4096, 4), (4096, 8))},
    **{f'{parts} parts of {heads * vdim} behind a state': (F, F.make_config([F.mamba_layer(heads=heads, vdim=vdim, state=8, groups=1, norm_groups=parts)] * 3, width=96))
       for heads, vdim, parts in ((2, 8, 1), (4, 16, 4), (32, 64, 1), (32, 64, 2), (32, 64, 8), (64, 64, 4), (64, 64, 8))},
}


@pytest.mark.parametrize('name', LONE)
def test_lone_rows(name):
    """A lone token's rows normed by the launches that read them, and (taps: every norm has a launch) by launches of their own: the same logits to the last bit."""
    cases, cfg = LONE[name]
    w = cases.random_weights(cfg, 5)
    mod = test_gpu_rofozen if cases is F else test_gpu_tolenex
    toks = mod.tokens_for(cfg, 200, 7)
    rows = [[s.step([('a', [t], [0])])[0] for t in toks] for s in (mod.session_for(cfg, w, 'bfloat16', max_sequences=1, debug_mode=mode) for mode in (False, True))]
    np.testing.assert_array_equal(*map(np.concatenate, rows))
