"""Wanted rows as they arrive in pinned memory, without a wait for the end of the stream: many steps on the same landing place, one row and several, rows of whole pieces and not,
ids alone, steps that outlast the wait for them (2 ms), more rows than the place takes, another stream from step to step."""
import numpy as np
import pytest
import torch

import rofozen_cases as F
import test_gpu_rofozen as G
from oracle import rofozen_oracle as O

pytestmark = pytest.mark.gpu


def small(vocab, width=32):
    return F.make_config([F.mamba_layer(heads=2, vdim=8, state=16, groups=1)], vocab=vocab, width=width)


@pytest.mark.parametrize('vocab', [211, 8192, 32003])
def test_many_steps(vocab):
    cfg = small(vocab)
    w = G.weights_for(cfg, 3, 'float32')
    s = G.session_for(cfg, w, 'float32', max_sequences=3)
    toks = {name: G.tokens_for(cfg, n, n) for name, n in (('a', 90), ('b', 60), ('c', 30))}
    got = G.replay(s, toks, [[(name, 1) for name, n in (('a', 90), ('b', 60), ('c', 30)) if at < n] for at in range(90)])
    for name, t in toks.items():
        G.check(got[name], O.logits(t, G.as_f64(w), cfg), G.F32_TOL, name)


def test_ids_alone():
    cfg = small(9001)
    w = G.weights_for(cfg, 3, 'float32')
    toks = G.tokens_for(cfg, 40, 5)
    rows = G.replay(G.session_for(cfg, w, 'float32'), {'a': toks}, [[('a', 1)]] * 40)['a']
    s = G.session_for(cfg, w, 'float32')
    for t, row in zip(toks, rows):
        none, ids = s.step([('a', [t], [0])], return_logits=False)
        assert none is None and ids.tolist() == [int(row.argmax())]


@pytest.mark.parametrize('rows', [1, 5, 700])
def test_a_long_step_and_many_rows(rows):
    """Products in plain fp32 FMAs: the step takes longer than rows are waited for.  700 rows of 8192 are more than the 8 MiB of the landing place.
    Bound: sums of up to 4096 terms in fp32, 2^-24 sqrt(4096) = 4e-6 a product by chance and 64 times that at worst, through two layers and the head."""
    cfg = F.make_config([F.mamba_layer(heads=2, vdim=8, state=16, groups=1, mlp=F.dense(ff=4096))] * 2, vocab=8192, width=768)
    w = G.weights_for(cfg, 3, 'float32')
    toks = G.tokens_for(cfg, 1500, 4)
    s = G.session_for(cfg, w, 'float32', max_tokens=2048)
    places = list(range(1500 - rows, 1500))
    logits, ids = s.step([('a', toks, places)])
    one, _ = s.step([('a', [7], [0])])
    want = O.logits(toks + [7], G.as_f64(w), cfg)
    G.check(logits, want[places], 1e-4, 'rows')
    G.check(one, want[1500:], 1e-4, 'the row behind them')
    np.testing.assert_array_equal(ids, logits.argmax(1))


def test_another_stream_from_step_to_step():
    cfg = small(211)
    w = G.weights_for(cfg, 3, 'float32')
    toks = G.tokens_for(cfg, 60, 6)
    s = G.session_for(cfg, w, 'float32')
    streams = [torch.cuda.Stream() for _ in range(3)]
    step, at = s.engine.step, []
    s.engine.step = lambda *a, **k: step(*a, **dict(k, stream=streams[len(at) % 3].cuda_stream))
    rows = []
    for t in toks:
        rows.append(s.step([('a', [t], [0])])[0])
        at.append(t)
    G.check(np.concatenate(rows), O.logits(toks, G.as_f64(w), cfg), G.F32_TOL)


def test_streams_in_turn_give_the_same_bits():
    """Steps that write and read states, caches and scratch of some size, on three streams in turn and on one."""
    cfg = F.make_config([F.mamba_layer(heads=16, vdim=64, state=64, groups=2, norm_groups=2, mlp=F.dense(ff=2048)), F.latent_layer(heads=8, dim=64, vdim=64, kv_rank=128, size=0)] * 2, width=1024, vocab=8192)
    w = F.random_weights(cfg, 3)
    toks, rows = G.tokens_for(cfg, 400, 6), ([1] * 9 + [31]) * 10
    streams, got = [torch.cuda.Stream() for _ in range(3)], []
    for many in (True, False):
        s = G.session_for(cfg, w, 'bfloat16')
        step, out, at = s.engine.step, [], 0
        for k, n in enumerate(rows):
            s.engine.step = lambda *a, **kw: step(*a, **dict(kw, stream=streams[k % 3 if many else 0].cuda_stream))
            out.append(s.step([('a', toks[at:at + n], [n - 1])])[0])
            at += n
        got.append(np.concatenate(out))
    np.testing.assert_array_equal(*got)
