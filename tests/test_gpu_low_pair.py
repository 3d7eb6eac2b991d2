"""The second halves of a delta layer's two low-rank pairs in one product of two (equal ranks, as many decays as outputs): ranks in whole pieces, of whole stages and of neither,
one row, a few and enough for tiles."""
import pytest

import narurax_cases as N
import test_gpu_narurax as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('rank', [3, 8, 64, 72])
def test_one_product_of_two(rank, dtype):
    cfg = N.make_config([N.delta_layer(heads=3, kv_heads=1, dim=16, vdim=16), N.delta_layer(heads=2, kv_heads=2, dim=24, vdim=24)])
    w = G.weights_for(cfg, 3, dtype, ranks=(rank, rank))
    toks = {'a': G.tokens_for(cfg, 56, 1), 'b': G.tokens_for(cfg, 9, 2)}
    got = G.replay(G.session_for(cfg, w, dtype), toks, [[('a', 1)], [('a', 1), ('b', 4)], [('a', 50)], [('a', 2), ('b', 3)], [('a', 1), ('b', 1)], [('a', 1)], [('b', 1)]])
    for name in toks:
        G.check_rows(got[name], toks[name], w, cfg, dtype, name)
