"""The token shift in the launch of the norm in front of it (steps of one row per entry): rows that end inside a wave, of a piece a thread and of two, and just outside the form
(no whole pieces of 4, longer than 8192); behind a dense result, behind experts; a sequence's first token, carries from prompts and from single rows, a slot that is used again."""
import pytest

import narurax_cases as N
import test_gpu_narurax as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('width', [96, 98, 260, 4096, 4100, 8192, 8196])
def test_steps_of_single_rows(width, dtype):
    small = dict(heads=2, kv_heads=1, dim=8, vdim=8)
    cfg = N.make_config([N.delta_layer(**small), N.delta_layer(mlp=N.moe(experts=4, top=2, ff=8), **small), N.delta_layer(**small)], width=width)
    w = G.weights_for(cfg, 3, dtype)
    s = G.session_for(cfg, w, dtype, max_sequences=2)
    for first, (a, b) in ((1, (7, 5)), (4, (8, 3))):
        toks = {f'a{first}': G.tokens_for(cfg, a, a), f'b{first}': G.tokens_for(cfg, b, b)}
        x, y = toks
        got = G.replay(s, toks, [[(x, first)], [(x, 1), (y, 1)], [(x, 1)], [(y, 1), (x, 1)]] + [[(y, b - 2)]] + [[(x, 1)]] * (a - first - 3))
        for name in toks:
            G.check_rows(got[name], toks[name], w, cfg, dtype, name)
