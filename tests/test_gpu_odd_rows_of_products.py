"""Products of 32 rows and more whose rows end inside a 128-byte stage (stack_gemm.hip: whole stages first, what is left of K added to the fp32 result):
one 16-byte piece, half a stage and all but a piece beyond whole stages, less than one stage, into a gated residual stream (Tolenex) and
into a plain fp32 result (Ruzinex's dense and shared feed-forward); rows at and beside a tile's edge.  Bounds as in the designs' own tests."""
import pytest

import ruzinex_cases as Z
import test_gpu_ruzinex as R
import test_gpu_tolenex as GT
import tolenex_cases as T

pytestmark = pytest.mark.gpu

LENGTHS = [56, 72, 96, 120, 264, 1048, 2104]


@pytest.mark.parametrize('rows', [32, 129])
@pytest.mark.parametrize('ff', LENGTHS)
def test_into_the_residual(ff, rows):
    cfg = T.make_config([T.attention_layer(heads=2, kv_heads=1, dim=64, vdim=128, rot_dims=64, ff=ff), T.hgrn2_layer(heads=2, dim=32, vdim=64, ff=ff)])
    w = T.random_weights(cfg, 41)
    toks = GT.tokens_for(cfg, rows, 42)
    got = T.replay(GT.session_for(cfg, w, 'bfloat16'), {'a': toks}, [[('a', rows)]])['a']
    GT.check_rows(got, toks, w, cfg, 'bfloat16', f'ff {ff}')


@pytest.mark.parametrize('rows', [32, 129])
@pytest.mark.parametrize('ff', LENGTHS)
@pytest.mark.parametrize('kind', ['dense', 'shared'])
def test_into_a_plain_result(kind, ff, rows):
    mlp = Z.dense(ff=ff) if kind == 'dense' else Z.moe(experts=3, top=3, ff=64, shared=ff)
    cfg = Z.make_config([Z.layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=mlp)], width=128)
    toks = R.tokens_for(cfg, rows, 43)
    w = R.weights_for(cfg, 44, 'bfloat16', toks)
    got = T.replay(R.session_for(cfg, w, 'bfloat16'), {'a': toks}, [[('a', rows)]])['a']
    R.check_rows(got, toks, w, cfg, 'bfloat16', f'ff {ff}')
