"""A lone token's normed row formed by the launch that reads it (stack_norm_impl.h: a mixer's or feed-forward's first product, the router's logits): rows of one
piece, that end inside a wave's quarter, of whole quarters and of the most a launch takes, and just outside the form (no whole pieces of 16, longer); the first row of a
stream, behind a dense feed-forward, behind experts, behind a shared expert; norms in 1, 2, 4 and 3 parts; few columns and very many; steps of more
tokens in between."""
import pytest

import rofozen_cases as F
import test_gpu_rofozen
import test_gpu_tolenex
import tolenex_cases as T

pytestmark = pytest.mark.gpu
STEPS = [[('a', k)] for k in (1, 1, 2, 1, 1)]
ROWS = sum(k for s in STEPS for _, k in s)


@pytest.mark.parametrize('dtype', ['bfloat16', 'float32'])
@pytest.mark.parametrize('width', [16, 96, 104, 512, 528, 1024, 1040, 2048, 2064, 4096, 4112])
def test_layers_on_one_stream(width, dtype):
    mod = test_gpu_rofozen
    mamba = dict(heads=2, vdim=16, state=16, groups=1, norm_groups=1)
    cfg = F.make_config([F.mamba_layer(mlp=F.dense(ff=40), **mamba), F.latent_layer(mlp=F.moe(experts=4, identity=2, top=2, count=1, keep=1)), F.mamba_layer(mlp=F.dense(ff=24), **mamba),
                         F.mamba_layer(mlp=None, **mamba), F.mamba_layer(mlp=F.moe(experts=3, identity=0, top=1, count=1, keep=1), **mamba)], width=width)
    toks = mod.tokens_for(cfg, ROWS, 7)
    w = mod.weights_for(cfg, 5, dtype, toks)
    mod.check_rows(mod.replay(mod.session_for(cfg, w, dtype), {'a': toks}, STEPS)['a'], toks, w, cfg, dtype)


@pytest.mark.parametrize('columns', [2, 2056])
def test_columns_of_the_first_product(columns):
    """2056 heads of 2 and more: more columns than 16 a CU, where a wave has whole rows."""
    mod = test_gpu_rofozen
    for width in (96, 1024, 2048, 2064):
        cfg = F.make_config([F.mamba_layer(heads=columns, vdim=2, state=8, groups=1, norm_groups=1, mlp=F.dense(ff=8))], width=width)
        toks = mod.tokens_for(cfg, ROWS, 7)
        w = F.random_weights(cfg, 5)
        mod.check_rows(mod.replay(mod.session_for(cfg, w, 'bfloat16'), {'a': toks}, STEPS)['a'], toks, w, cfg, 'bfloat16')


@pytest.mark.parametrize('width,groups', [(96, 1), (96, 2), (96, 4), (96, 3), (1040, 2), (1040, 4), (2048, 4), (4096, 1), (4096, 4), (4112, 4)])
def test_norms_in_parts(width, groups):
    """... which also leave the row that the feed-forward reads; layers without one."""
    mod = test_gpu_tolenex
    cfg = T.make_config([T.attention_layer(heads=2, kv_heads=1, dim=16, vdim=16, rot_dims=8, ff=40), T.hgrn2_layer(heads=2, dim=16, vdim=16, ff=24),
                         T.attention_layer(heads=2, kv_heads=1, dim=16, vdim=16, rot_dims=8, ff=0)], width=width, groups=groups)
    toks = mod.tokens_for(cfg, ROWS, 7)
    w = T.random_weights(cfg, 5)
    mod.check_rows(T.replay(mod.session_for(cfg, w, 'bfloat16'), {'a': toks}, STEPS)['a'], toks, w, cfg, 'bfloat16')
