"""Steps of one token whose experts' products choose for themselves (stack_gemm.hip lone_up_kernel, choose_in_wave): one output and as many as a wave
has lanes, and one more (which takes the ordering launch); 8 choices, and more (which take it too); groups; identities; every output chosen; equal scores
(the lowest outputs win); rows of less than a chunk and of several; the choice by softmax and by sigmoid, biased and corrected, weights on the input and
on the output, a shared expert beside; and steps of more tokens in between."""
import numpy as np
import pytest

import narurax_cases
import rofozen_cases
import ruzinex_cases
import test_gpu_narurax
import test_gpu_rofozen
import test_gpu_ruzinex

pytestmark = pytest.mark.gpu

STEPS = [[('a', k)] for k in (1, 1, 2, 1)]
ROUTERS = [dict(experts=1, identity=0, top=1, count=1, keep=1), dict(experts=6, identity=3, top=2, count=3, keep=2), dict(experts=17, identity=0, top=3, count=1, keep=1),
           dict(experts=60, identity=4, top=2, count=8, keep=3), dict(experts=64, identity=0, top=64, count=1, keep=1), dict(experts=64, identity=0, top=8, count=1, keep=1),
           dict(experts=5, identity=3, top=8, count=1, keep=1), dict(experts=65, identity=0, top=3, count=1, keep=1)]


def run(mod, cfg, w, toks):
    mod.check_rows(mod.replay(mod.session_for(cfg, w, 'bfloat16'), {'a': toks}, STEPS)['a'], toks, w, cfg, 'bfloat16')


@pytest.mark.parametrize('equal', [False, True], ids=['apart', 'equal'])
@pytest.mark.parametrize('width,ff', [(72, 8), (1032, 520)])
@pytest.mark.parametrize('router', ROUTERS, ids=lambda r: f"{r['experts']}+{r['identity']}top{r['top']}")
def test_corrected_softmax_and_identities(router, width, ff, equal):
    Z, mod = rofozen_cases, test_gpu_rofozen
    cfg = Z.make_config([Z.mamba_layer(mlp=Z.moe(ff=ff, **router))] * (2 if router['experts'] < 20 else 1), width=width)
    toks = mod.tokens_for(cfg, sum(n for s in STEPS for _, n in s), 7)
    if equal or router['experts'] > 20:  # (among many outputs a random choice is always close: the corrections alone decide)
        w = Z.random_weights(cfg, 5)
        for name in w:
            if name.endswith('mlp.router'):
                w[name] = np.zeros_like(w[name])
            if name.endswith('mlp.correction'):
                n = len(w[name])
                w[name] = np.zeros_like(w[name]) if equal else (np.random.default_rng(3).permutation(n) / n).astype(w[name].dtype)
    else:
        w = mod.weights_for(cfg, 5, 'bfloat16', toks)
    run(mod, cfg, w, toks)


@pytest.mark.parametrize('experts,top', [(1, 1), (11, 4), (8, 8), (9, 9)])
@pytest.mark.parametrize('width,ff', [(72, 8), (1032, 520)])
def test_sigmoid_and_input_weights(experts, top, width, ff):
    Z, mod = narurax_cases, test_gpu_narurax
    moe = Z.moe(experts=experts, top=top, ff=ff)
    cfg = Z.make_config([Z.attn_layer(mlp=moe)] * (2 if experts < 20 else 1), width=width)
    toks = mod.tokens_for(cfg, sum(n for s in STEPS for _, n in s), 7)
    run(mod, cfg, mod.weights_for(cfg, 5, 'bfloat16', toks), toks)


@pytest.mark.parametrize('experts,top', [(1, 1), (11, 4), (64, 2), (65, 2)])
@pytest.mark.parametrize('width,ff,shared', [(72, 8, 16), (1032, 520, 0)])
def test_biased_softmax_and_a_shared_expert(experts, top, width, ff, shared):
    Z, mod = ruzinex_cases, test_gpu_ruzinex
    cfg = Z.make_config([Z.layer(mlp=Z.moe(experts=experts, top=top, ff=ff, shared=shared))] * (2 if experts < 20 else 1), width=width)
    toks = mod.tokens_for(cfg, sum(n for s in STEPS for _, n in s), 7)
    run(mod, cfg, mod.weights_for(cfg, 5, 'bfloat16', toks), toks)
