"""Router of a few tokens in one launch (stack_moe.hip moe_route_few_kernel): logits spread over workgroups, the last of them chooses and
orders.  Outputs that end inside a workgroup or take many of them, more than 64 choices' worth of lanes, groups, equal scores (the lowest
outputs win), rows that are not whole 16-byte pieces, and 1, 7, 8 and 9 tokens (the most the launch takes, and one more), several steps
in a row so that its ticket is armed again each time."""
import numpy as np
import pytest

from rofozen_cases import make_config, mamba_layer, moe, random_weights
from test_gpu_rofozen import O, as_f64, check, replay, session_for, tokens_for, tol_of

pytestmark = pytest.mark.gpu

ROUTERS = [dict(experts=1, identity=0, top=1, count=1, keep=1), dict(experts=6, identity=3, top=2, count=3, keep=2), dict(experts=17, identity=0, top=5, count=1, keep=1),
           dict(experts=150, identity=10, top=7, count=8, keep=3), dict(experts=70, identity=0, top=64, count=1, keep=1)]


@pytest.mark.parametrize('equal', [False, True], ids=['apart', 'equal'])
@pytest.mark.parametrize('width', [96, 100])
@pytest.mark.parametrize('router', ROUTERS, ids=lambda r: f"{r['experts']}+{r['identity']}top{r['top']}")
def test_few_token_router(router, width, equal):
    cfg = make_config([mamba_layer(mlp=moe(ff=8, **router)), mamba_layer(mlp=moe(ff=8, **router))], width=width)
    w = random_weights(cfg, 5)
    if equal:  # every output's score is the same number: the first ones are chosen
        for name in w:
            if name.endswith(('mlp.router', 'mlp.correction')):
                w[name] = np.zeros_like(w[name])
    toks = tokens_for(cfg, 29, 7)
    got = replay(session_for(cfg, w, 'float32'), {'a': toks}, [[('a', k)] for k in (1, 7, 8, 9, 1, 1, 2)])['a']
    check(got, O.logits(toks, as_f64(w), cfg), tol_of('float32'), 'a')


@pytest.mark.parametrize('n', [256, 257, 300])
@pytest.mark.parametrize('router', [ROUTERS[1], ROUTERS[2], ROUTERS[3]], ids=lambda r: f"{r['experts']}+{r['identity']}")
@pytest.mark.parametrize('width', [96, 128, 1056])
def test_prompt_router(width, router, n):
    """Logits of prompts through fp32 matrix products (from 257 tokens on, widths of whole 32-value pieces): tokens and outputs that end inside
    a tile, widths shorter than the waves' first round and longer."""
    cfg = make_config([mamba_layer(mlp=moe(ff=8, **router))], width=width)
    w = random_weights(cfg, 6)
    toks = tokens_for(cfg, n, 8)
    got = replay(session_for(cfg, w, 'float32'), {'a': toks}, [[('a', n)]])['a']
    check(got, O.logits(toks, as_f64(w), cfg), tol_of('float32'), 'a')


def test_the_most_outputs_and_tokens_of_one_launch():
    """1024 outputs, 8 tokens: scores and choice values are 64 KiB of LDS, and the launch's ticket comes on top."""
    cfg = make_config([mamba_layer(mlp=moe(experts=1000, identity=24, top=3, count=1, keep=1, ff=8))], width=64)
    w = random_weights(cfg, 9)
    toks = tokens_for(cfg, 16, 10)
    got = replay(session_for(cfg, w, 'float32'), {'a': toks}, [[('a', 8)], [('a', 7)], [('a', 1)]])['a']
    check(got, O.logits(toks, as_f64(w), cfg), tol_of('float32'), 'a')
