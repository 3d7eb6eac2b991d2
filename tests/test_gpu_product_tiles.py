"""The bfloat16 products of many rows (launch_glds_bf16 of stack_gemm.hip) in every tile shape they choose from: K of one stage of 128 bytes, of as
many as the stages' ring holds, of one more and of three rings; rows and columns that end inside a tile; columns that do and do not leave
in 16-byte pieces; plain, gated and grouped products and the gated residual.  Which sizes take which shape is what
test_stack_host_runtime.py checks, without a GPU."""
import numpy as np
import pytest

import ruzinex_cases as Z
import test_gpu_ruzinex as R
import test_gpu_tolenex
import tolenex_cases as T

pytestmark = pytest.mark.gpu

ROWS = 1000
# tile shape: (columns of a plain product, ff of a gated one, ff of two grouped ones) that take it at 1000 rows on 256 CUs
SHAPES = {(128, 64): (2004, 1000, 504), (128, 128): (4004, 2000, 1000), (128, 192): (6004, 3000, 1472), (128, 256): (8004, 4000, 1984),
          (256, 192): (12004, 6000, 3008), (256, 256): (16004, 8000, 4032)}
FEW = {(128, 256): (8, 2), (128, 128): (40, 2)}  # experts, choices: groups of 250 and of 50 rows on average
RESIDUAL = {(128, 64): (1000, 512), (128, 128): (1000, 2112), (128, 192): (2000, 3072)}  # rows, width


def plain_config(columns, k):
    return Z.make_config([Z.layer(heads=2, kv_heads=1, dim=32, vdim=32)], width=k, vocab=columns)


def gated_config(mlp, k):
    return Z.make_config([Z.layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=mlp)], width=k)


def residual_config(width):
    return T.make_config([T.attention_layer(heads=4, kv_heads=1, dim=32, vdim=64, rot_dims=16, ff=320)], width=width, groups=2)


def plain(columns, k):
    """The head's product against 64-bit sums over the rows it reads: the engine's residual stream behind its layer, normed and rounded here.  A
    value of a row may be rounded the other way, by 2^-8 of itself at most; the fp32 sums add K 2^-24."""
    cfg = plain_config(columns, k)
    toks = R.tokens_for(cfg, ROWS, 5)
    w = Z.random_weights(cfg, 6)
    s = R.session_for(cfg, w, 'bfloat16', debug_mode=True)
    got, _ = s.step([('a', toks, list(range(ROWS)))])
    x = s.engine.tap(0).astype(np.float64)
    h = R.to_bf16(x / np.sqrt((x * x).mean(1, keepdims=True) + cfg['norm']['eps']) * w['final.norm'])
    want = h @ w['embed'].astype(np.float64).T
    e = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert (e < 2.0 ** -8 + k * 2.0 ** -24).all(), f'row {int(e.argmax())} is off by {e.max():.3g}'
    worst = np.abs(got - want) / (np.abs(h) @ np.abs(w['embed'].astype(np.float64)).T)
    assert (worst < 2.0 ** -8 + k * 2.0 ** -24).all(), f'place {np.unravel_index(worst.argmax(), worst.shape)} is off by {worst.max():.3g} of its terms'


@pytest.mark.parametrize('k', [64, 128, 192, 256, 320, 832])
@pytest.mark.parametrize('shape', sorted(SHAPES), ids=str)
def test_plain_product(shape, k):
    plain(SHAPES[shape][0], k)


@pytest.mark.parametrize('shape', sorted(SHAPES), ids=str)
def test_plain_product_of_odd_columns(shape):
    plain(SHAPES[shape][0] - 1, 320)


@pytest.mark.parametrize('k', [64, 320, 576])
@pytest.mark.parametrize('shape', sorted(SHAPES), ids=str)
def test_gated_product(shape, k):
    cfg = gated_config(Z.dense(ff=SHAPES[shape][1]), k)
    toks = R.tokens_for(cfg, ROWS, 97)
    w = Z.random_weights(cfg, 98)
    R.check_rows(R.replay(R.session_for(cfg, w, 'bfloat16'), {'a': toks}, [[('a', ROWS)]])['a'], toks, w, cfg, 'bfloat16')


@pytest.mark.parametrize('k', [64, 320, 576])
@pytest.mark.parametrize('shape', sorted(SHAPES), ids=str)
def test_grouped_product(shape, k):
    cfg = gated_config(Z.moe(experts=2, top=2, ff=SHAPES[shape][2], shared=0), k)
    toks = R.tokens_for(cfg, ROWS, 97)
    w = Z.random_weights(cfg, 98)
    R.check_rows(R.replay(R.session_for(cfg, w, 'bfloat16'), {'a': toks}, [[('a', ROWS)]])['a'], toks, w, cfg, 'bfloat16')


@pytest.mark.parametrize('k', [64, 320])
@pytest.mark.parametrize('shape', sorted(FEW), ids=str)
def test_grouped_product_of_small_groups(shape, k):
    experts, top = FEW[shape]
    cfg = gated_config(Z.moe(experts=experts, top=top, ff=192, shared=0), k)
    toks = R.tokens_for(cfg, ROWS, 97)
    w = R.weights_for(cfg, 98, 'bfloat16', toks)
    R.check_rows(R.replay(R.session_for(cfg, w, 'bfloat16'), {'a': toks}, [[('a', ROWS)]])['a'], toks, w, cfg, 'bfloat16')


@pytest.mark.parametrize('rows,width', sorted(RESIDUAL.values()) + [(1000, 1030)])
def test_gated_residual(rows, width):
    """Both of a layer's sublayers land through a gate with a bias; a width of 1030 leaves value by value."""
    cfg = residual_config(width)
    toks = test_gpu_tolenex.tokens_for(cfg, rows, 5)
    w = T.random_weights(cfg, 6)
    s = test_gpu_tolenex.session_for(cfg, w, 'bfloat16', max_tokens=2048)
    test_gpu_tolenex.check_rows(T.replay(s, {'a': toks}, [[('a', rows)]])['a'], toks, w, cfg, 'bfloat16')
