"""Steps of single decoded tokens: the recurrences' one-row launches (stack_ssm.hip ssm_step_kernel, stack_delta.hip delta_step_kernel) at shapes of
one thread, of threads that do not fill a wave, of the largest state a workgroup holds and just outside the form (rows not a multiple of
8, columns not of 4), fresh and carried states, one to five requests; and the 16-byte forms of the embedding and the latent queries'
norm at one and several pieces per thread; and the convolution of prompts in runs of rows."""
import numpy as np
import pytest

import narurax_cases
import rofozen_cases
import test_gpu_narurax
import test_gpu_rofozen
from test_gpu_chunked_recurrences import KINDS

pytestmark = pytest.mark.gpu

SHAPES = {'mamba2': [(8, 4), (8, 12), (24, 20), (128, 64), (512, 64), (64, 256), (12, 8), (16, 6)],
          'delta': [(8, 4), (24, 12), (40, 36), (128, 128), (512, 32), (256, 128), (12, 8), (16, 6)]}


@pytest.mark.parametrize('dtype', ['bfloat16', 'float32'])
@pytest.mark.parametrize('kind,dim,vdim', [(k, d, v) for k in SHAPES for d, v in SHAPES[k]])
def test_one_row_recurrences(kind, dim, vdim, dtype):
    mod, cfg, _ = KINDS[kind](dim, vdim)
    reqs = {r: mod.tokens_for(cfg, 7, 3 + i) for i, r in enumerate('abcde')}
    w = mod.random_weights(cfg, 11)
    steps = [[('a', 1)]] * 3 + [[('a', 1), ('b', 1)]] * 2 + [[(r, 1) for r in 'bcde']] + [[('c', 3), ('a', 1)]] + [[(r, 1) for r in 'abcde']]
    n = {r: sum(k for s in steps for q, k in s if q == r) for r in reqs}
    reqs = {r: t[:n[r]] for r, t in reqs.items()}
    got = mod.replay(mod.session_for(cfg, w, dtype, max_sequences=5), reqs, steps)
    for r, toks in reqs.items():
        if kind == 'mamba2':
            mod.check(got[r], mod.O.logits(toks, mod.as_f64(w), cfg), mod.tol_of(dtype), r)
        else:
            mod.check_rows(got[r], toks, w, cfg, dtype, r)


@pytest.mark.parametrize('dtype', ['bfloat16', 'float32'])
@pytest.mark.parametrize('conv,vdim,state', [(4, 12, 10), (4, 13, 10), (3, 12, 10), (5, 12, 10), (4, 64, 32)])
def test_convolution_runs(conv, vdim, state, dtype):
    """stack_ssm.hip ssm_conv_run_kernel (4 taps, from 64 rows on, channels in whole fours): runs that cross entries, entries shorter than the
    taps beside long ones, portions that carry the tail in and out, and the shapes just outside the form."""
    mod = test_gpu_rofozen
    cfg = rofozen_cases.make_config([rofozen_cases.mamba_layer(heads=4, groups=2, vdim=vdim, state=state, conv=conv, norm_groups=2)])
    w = rofozen_cases.random_weights(cfg, 4)
    steps = [[('a', 63)], [('a', 1), ('b', 2), ('c', 61)], [('b', 1), ('a', 33), ('c', 3), ('d', 70)], [('d', 64)], [('a', 2), ('d', 65), ('b', 9)]]
    reqs = {r: mod.tokens_for(cfg, sum(k for s in steps for q, k in s if q == r), 3 + i) for i, r in enumerate('abcd')}
    got = mod.replay(mod.session_for(cfg, w, dtype), reqs, steps)
    for r, toks in reqs.items():
        # (a row's bound in bfloat16: what rounding the oracle's own activations does to it; a flat one fails where a group's outputs cancel)
        mod.check_rows(got[r], toks, w, cfg, dtype, r)


@pytest.mark.parametrize('width,q_rank', [(96, 8), (104, 2048), (2056, 2056), (100, 28), (40, 8200)])
def test_embedding_and_latent_norm(width, q_rank):
    mod = test_gpu_rofozen
    cfg = rofozen_cases.make_config([rofozen_cases.latent_layer(q_rank=q_rank)], width=width)
    w = rofozen_cases.random_weights(cfg, 4)
    toks = mod.tokens_for(cfg, 9, 6)
    got = mod.replay(mod.session_for(cfg, w, 'float32'), {'a': toks}, [[('a', 5)]] + [[('a', 1)]] * 4)['a']
    mod.check(got, mod.O.logits(toks, mod.as_f64(w), cfg), mod.tol_of('float32'), 'a')
