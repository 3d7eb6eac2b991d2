"""Products of one row (row_kernel of stack_gemm.hip): K of less than one 512-column chunk, of whole chunks and one 16-byte piece more at every number
of chunks per wave and of waves per row, beyond the longest row that is requested at once; odd columns, and columns enough that a wave has rows of its
own; the plain (against an exactly known row), gated, grouped and residual epilogues.  Bounds of the others as in the designs' own tests."""
import numpy as np
import pytest

import rofozen_cases as M
import ruzinex_cases as Z
import test_gpu_rofozen as RF
import test_gpu_ruzinex as R
import test_gpu_tolenex as GT
import tolenex_cases as T
from test_gpu_slim_shapes import check_head, known_rows

pytestmark = pytest.mark.gpu

ONE = [[('a', 1)]] * 3
LENGTHS = [8, 504, 512, 520, 1024, 1032, 1536, 1544, 2048, 2056, 4096, 4104, 6144, 6152, 8192, 8200, 12288, 12296]


@pytest.mark.parametrize('k', LENGTHS)
@pytest.mark.parametrize('columns', [37, 4101])
def test_plain_product(columns, k):
    s, toks, h, w = known_rows(columns, k, 1)
    got, _ = s.step([('a', toks, [0])])
    np.testing.assert_array_equal(s.engine.tap(0), w[:1])
    check_head(got, h, w)


@pytest.mark.parametrize('k', [8, 72, 256, 264, 504, 512])
@pytest.mark.parametrize('columns', [10761, 16387])
def test_short_rows_of_many_columns(columns, k):
    test_plain_product(columns, k)


@pytest.mark.parametrize('heads,dim,kv_rank', [(64, 16, 171), (128, 32, 88), (64, 260, 258)])
def test_short_rows_of_many_heads(heads, dim, kv_rank):
    cfg = M.make_config([M.latent_layer(heads=heads, dim=dim, vdim=16, kv_rank=kv_rank)])
    toks = RF.tokens_for(cfg, 3, 97)
    w = M.random_weights(cfg, 98)
    RF.check_rows(RF.replay(RF.session_for(cfg, w, 'bfloat16'), {'a': toks}, ONE)['a'], toks, w, cfg, 'bfloat16')


@pytest.mark.parametrize('k,ff', [(72, 504), (520, 1032), (1032, 1536), (1544, 2056), (2056, 520), (4104, 64)])
@pytest.mark.parametrize('kind', ['dense', 'moe', 'shared'])
def test_gated_and_grouped_products(kind, k, ff):
    mlp = {'dense': Z.dense(ff=ff), 'moe': Z.moe(experts=70, top=3, ff=ff, shared=0), 'shared': Z.moe(experts=3, top=2, ff=ff, shared=ff)}[kind]
    cfg = Z.make_config([Z.layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=mlp)], width=k, vocab=61)
    toks = R.tokens_for(cfg, 3, 97)
    w = R.weights_for(cfg, 98, 'bfloat16', toks)
    R.check_rows(R.replay(R.session_for(cfg, w, 'bfloat16'), {'a': toks}, ONE)['a'], toks, w, cfg, 'bfloat16')


@pytest.mark.parametrize('k,ff', [(2056, 8), (2560, 72), (2056, 136), (3072, 136), (256, 176)])
def test_rows_of_a_few_chunks_through_many_groups(k, ff):
    cfg = Z.make_config([Z.layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=Z.moe(experts=65, top=32, ff=ff, shared=0))], width=k, vocab=61)
    toks = R.tokens_for(cfg, 3, 97)
    w = R.weights_for(cfg, 98, 'bfloat16', toks)
    R.check_rows(R.replay(R.session_for(cfg, w, 'bfloat16'), {'a': toks}, ONE)['a'], toks, w, cfg, 'bfloat16')


@pytest.mark.parametrize('width,ff', [(1000, 512), (1000, 2120), (2000, 3080)])
def test_gated_residual(width, ff):
    cfg = T.make_config([T.attention_layer(heads=4, kv_heads=1, dim=32, vdim=64, rot_dims=16, ff=ff)], width=width, groups=2)
    toks = GT.tokens_for(cfg, 3, 7)
    w = T.random_weights(cfg, 8)
    GT.check_rows(T.replay(GT.session_for(cfg, w, 'bfloat16'), {'a': toks}, ONE)['a'], toks, w, cfg, 'bfloat16')
