"""A lone token's state-space output normed by the out-projection that reads it: parts of a row that end where a wave does and, 8 of them, in the middle of one; rows that
are refused (parts and lengths that fit neither, no whole pieces of 16, longer than 4096); few columns and many; steps of more tokens in between.  8 parts of a residual row, too."""
import pytest

import rofozen_cases as F
import test_gpu_lone_norm as L
import test_gpu_rofozen
import test_gpu_tolenex
import tolenex_cases as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', ['bfloat16', 'float32'])
@pytest.mark.parametrize('heads,vdim,parts', [(2, 8, 1), (4, 16, 4), (4, 18, 4), (6, 16, 3), (8, 64, 8), (16, 64, 8), (32, 64, 1), (32, 64, 2), (32, 64, 8), (32, 96, 8), (64, 64, 4), (64, 64, 8),
                                              (64, 66, 8)])
def test_rows_and_parts(heads, vdim, parts, dtype):
    mod = test_gpu_rofozen
    for width in (32, 2100):
        cfg = F.make_config([F.mamba_layer(heads=heads, vdim=vdim, state=8, groups=1, norm_groups=parts), F.mamba_layer(heads=heads, vdim=vdim, state=8, groups=2, norm_groups=parts)], width=width)
        toks = mod.tokens_for(cfg, L.ROWS, 7)
        w = F.random_weights(cfg, 5)
        mod.check_rows(mod.replay(mod.session_for(cfg, w, dtype), {'a': toks}, L.STEPS)['a'], toks, w, cfg, dtype)


@pytest.mark.parametrize('width', [1024, 2048, 4096])
def test_eight_parts_of_the_residual(width):
    mod = test_gpu_tolenex
    cfg = T.make_config([T.attention_layer(heads=2, kv_heads=1, dim=16, vdim=16, rot_dims=8, ff=40), T.hgrn2_layer(heads=2, dim=16, vdim=16, ff=24)], width=width, groups=8)
    toks = mod.tokens_for(cfg, L.ROWS, 7)
    w = T.random_weights(cfg, 5)
    mod.check_rows(T.replay(mod.session_for(cfg, w, 'bfloat16'), {'a': toks}, L.STEPS)['a'], toks, w, cfg, 'bfloat16')
