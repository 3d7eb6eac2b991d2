"""Products of one row (row_kernel of stack_gemm.hip): K of less than one 512-column chunk, of whole chunks and one 16-byte piece more at every number
of chunks per wave and of waves per row, beyond the longest row that is requested at once; odd columns, and columns enough that a wave has rows of its
own; the plain, gated, grouped and residual epilogues.  Bounds as in test_gpu_product_tiles."""
import numpy as np
import pytest

import ruzinex_cases as Z
import test_gpu_ruzinex as R
import test_gpu_tolenex as GT
import tolenex_cases as T

pytestmark = pytest.mark.gpu

ONE = [[('a', 1)]] * 3
LENGTHS = [8, 504, 512, 520, 1024, 1032, 1536, 1544, 2048, 2056, 4096, 4104, 6144, 6152, 8192, 8200, 12288, 12296]


@pytest.mark.parametrize('k', LENGTHS)
@pytest.mark.parametrize('columns', [37, 4101])
def test_plain_product(columns, k):
    cfg = Z.make_config([Z.layer(heads=2, kv_heads=1, dim=32, vdim=32)], width=k, vocab=columns)
    toks = R.tokens_for(cfg, 1, 5)
    w = Z.random_weights(cfg, 6)
    s = R.session_for(cfg, w, 'bfloat16', debug_mode=True)
    got, _ = s.step([('a', toks, [0])])
    x = s.engine.tap(0).astype(np.float64)
    h = R.to_bf16(x / np.sqrt((x * x).mean(1, keepdims=True) + cfg['norm']['eps']) * w['final.norm'])
    want = h @ w['embed'].astype(np.float64).T
    e = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert (e < 2.0 ** -8 + k * 2.0 ** -24).all(), f'off by {e.max():.3g}'
    worst = np.abs(got - want) / (np.abs(h) @ np.abs(w['embed'].astype(np.float64)).T)
    assert (worst < 2.0 ** -8 + k * 2.0 ** -24).all(), f'place {worst.argmax()} is off by {worst.max():.3g} of its terms'


@pytest.mark.parametrize('k,ff', [(72, 504), (520, 1032), (1032, 1536), (1544, 2056), (2056, 520), (4104, 64)])
@pytest.mark.parametrize('kind', ['dense', 'moe', 'shared'])
def test_gated_and_grouped_products(kind, k, ff):
    mlp = {'dense': Z.dense(ff=ff), 'moe': Z.moe(experts=70, top=3, ff=ff, shared=0), 'shared': Z.moe(experts=3, top=2, ff=ff, shared=ff)}[kind]
    cfg = Z.make_config([Z.layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=mlp)], width=k, vocab=61)
    toks = R.tokens_for(cfg, 3, 97)
    w = R.weights_for(cfg, 98, 'bfloat16', toks)
    R.check_rows(R.replay(R.session_for(cfg, w, 'bfloat16'), {'a': toks}, ONE)['a'], toks, w, cfg, 'bfloat16')


@pytest.mark.parametrize('width,ff', [(1000, 512), (1000, 2120), (2000, 3080)])
def test_gated_residual(width, ff):
    cfg = T.make_config([T.attention_layer(heads=4, kv_heads=1, dim=32, vdim=64, rot_dims=16, ff=ff)], width=width, groups=2)
    toks = GT.tokens_for(cfg, 3, 7)
    w = T.random_weights(cfg, 8)
    GT.check_rows(T.replay(GT.session_for(cfg, w, 'bfloat16'), {'a': toks}, ONE)['a'], toks, w, cfg, 'bfloat16')
