"""The start of a step in one launch (metadata, embedding, pair embedding): one token, the most that it takes and one more, rows of one piece, of more than a workgroup has and
of no whole pieces; a sequence's first token and later ones; a looped stack, which keeps the rows."""
import pytest

import narurax_cases as N
import test_gpu_narurax
import test_gpu_tolenex
import tolenex_cases as T

pytestmark = pytest.mark.gpu
STEPS = [[('a', 16)], [('a', 1), ('b', 15)], [('a', 17)], [('a', 1), ('b', 2)], [('a', 1)], [('b', 1), ('a', 1)]]


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('width', [8, 96, 100, 2056])
def test_pair_embedding(width, dtype):
    cfg = N.make_config([N.delta_layer(heads=2, kv_heads=1, dim=8, vdim=8)], width=width)
    w = test_gpu_narurax.weights_for(cfg, 3, dtype)
    toks = {'a': test_gpu_narurax.tokens_for(cfg, 37, 1), 'b': test_gpu_narurax.tokens_for(cfg, 18, 2)}
    got = test_gpu_narurax.replay(test_gpu_narurax.session_for(cfg, w, dtype), toks, STEPS)
    for name in toks:
        test_gpu_narurax.check_rows(got[name], toks[name], w, cfg, dtype, name)


@pytest.mark.parametrize('width', [96, 100])
def test_looped_stack(width):
    layers = [T.attention_layer(heads=2, kv_heads=1, dim=16, vdim=16, rot_dims=8, ff=40), T.hgrn2_layer(heads=2, dim=16, vdim=16, ff=24)]
    cfg = T.make_config(layers, width=width, groups=2, loop=(0, 2, 2))
    w = T.random_weights(cfg, 5)
    toks = {'a': test_gpu_tolenex.tokens_for(cfg, 37, 1), 'b': test_gpu_tolenex.tokens_for(cfg, 18, 2)}
    got = T.replay(test_gpu_tolenex.session_for(cfg, w, 'bfloat16'), toks, STEPS)
    for name in toks:
        test_gpu_tolenex.check_rows(got[name], toks[name], w, cfg, 'bfloat16', name)
