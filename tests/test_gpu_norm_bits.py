"""Norms to the last bit: the fp32 sum of squares in the order that its launch has (a lane's four squares, a tree over 64 lanes, the waves in turn), which the order of the
compiler's own contractions would otherwise change with the code around it.  A value of a normed bfloat16 row turns over one time in 30000 where its row's sum is another in
the last bit: rows enough that this shows, which each test asks of its inputs first."""
import numpy as np
import pytest

import narurax_cases as N
import test_gpu_narurax
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
