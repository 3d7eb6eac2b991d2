"""The tiles of 128 rows and 16 x 16 MFMAs of gemm_wide_impl.h: the forms that test_gpu_product_tiles.py does not reach.  fp32 rows in whole pieces with K of one
stage, of as many as the ring holds, of one more and of three rings; fp32 sections of 16 columns and of one behind gated columns, of the 256 x 256 tiles too; the
fp32 residual without a gate, and with one in tiles of 256 columns; how a gated result is rounded.  Which sizes take which shape is what test_stack_host_runtime.py checks, without a GPU."""
import numpy as np
import pytest

import ruzinex_cases as Z
import sodudra_cases as S
import test_gpu_product_tiles as P
import test_gpu_ruzinex as R
import test_gpu_sodudra
import test_gpu_tolenex
import test_gpu_wide_tiles as W
import tolenex_cases as T

pytestmark = pytest.mark.gpu

# tile shape: columns of a plain product at 1000 rows, ff of a shared expert beside 16 experts' logits and a gate, (rows, width) of a residual
COLUMNS = {(128, 64): 2000, (128, 128): 4000, (128, 192): 6000, (128, 256): 8000}
SHARED = {(128, 64): 1000, (128, 128): 2000, (128, 192): 3000, (128, 256): 4000}
WIDE_SHARED = (8000, 2496)                                      # ff, width
RESIDUAL = {(128, 64): (1000, 512), (128, 128): (1000, 2112), (128, 192): (2000, 3072), (128, 256): (2000, 4096)}


def shared_config(ff, width=320):
    return P.gated_config(Z.moe(experts=16, top=2, ff=32, shared=ff), width)


def residual_config(width):
    return S.make_config([S.layer(heads=4, dim=32, vdim=32, kv_rank=64, mlp=S.moe(experts=2, top=1, ff=32, shared=320 - 4 * 32))], width=width, side=0)


@pytest.mark.parametrize('k', [64, 192, 256, 320, 832])
@pytest.mark.parametrize('shape', sorted(COLUMNS), ids=str)
def test_rows_in_whole_pieces(shape, k):
    P.plain(COLUMNS[shape], k)


@pytest.mark.parametrize('ff,width', [(ff, 320) for ff in SHARED.values()] + [WIDE_SHARED])
def test_narrow_sections(ff, width):
    cfg = shared_config(ff, width)
    toks = R.tokens_for(cfg, P.ROWS, 97)
    w = R.weights_for(cfg, 98, 'bfloat16', toks)
    R.check_rows(R.replay(R.session_for(cfg, w, 'bfloat16'), {'a': toks}, [[('a', P.ROWS)]])['a'], toks, w, cfg, 'bfloat16')


@pytest.mark.parametrize('rows,width', sorted(RESIDUAL.values()))
def test_residual(rows, width):
    cfg = residual_config(width)
    toks = test_gpu_sodudra.tokens_for(cfg, rows, 5)
    w = S.random_weights(cfg, 6)
    s = test_gpu_sodudra.session_for(cfg, w, 'bfloat16', max_tokens=2048)
    test_gpu_sodudra.check_rows(T.replay(s, {'a': toks}, [[('a', rows)]])['a'], toks, w, cfg, 'bfloat16')


def test_gated_residual():
    rows, width = RESIDUAL[128, 256]
    cfg = P.residual_config(width)
    toks = test_gpu_tolenex.tokens_for(cfg, rows, 5)
    w = T.random_weights(cfg, 6)
    s = test_gpu_tolenex.session_for(cfg, w, 'bfloat16', max_tokens=2048)
    test_gpu_tolenex.check_rows(T.replay(s, {'a': toks}, [[('a', rows)]])['a'], toks, w, cfg, 'bfloat16')


@pytest.mark.parametrize('rows,cfg', [(rows, P.residual_config(width)) for rows, width in sorted(RESIDUAL.values())] + [(W.RESIDUAL[0], W.residual_config(T))],
                         ids=[*map(str, sorted(RESIDUAL)), '256 x 256'])
def test_gate_and_residual_round_apart(rows, cfg):
    """x + g v as two operations in fp32, the same bits by every tile.  The second matrix picks one value v of a row for columns n and n + half, and x is zero in the second
    half, which then holds g v as it was rounded."""
    half, width, ff = cfg['width'] // 2, cfg['width'], cfg['layers'][0]['mlp']['ff']
    w = T.random_weights(cfg, 6)
    columns = np.arange(width)
    w['embed'][:, half:] = 0
    w['l0.mix.o'][:] = w['l0.rg2'][:] = w['l0.mlp.down'][:] = 0
    w['l0.mlp.down'][columns, columns % half % ff] = 1
    w['l0.rg2.b'][:] = 0.3125
    toks = test_gpu_tolenex.tokens_for(cfg, rows, 5)
    s = test_gpu_tolenex.session_for(cfg, w, 'bfloat16', max_tokens=4096, max_batch_tokens=4096, max_sequences=1, debug_mode=True)
    s.step([('a', toks, [0])])
    x, scaled = w['embed'][toks, :half] * np.float32(cfg['embedding']['scale']), s.engine.tap(0)
    apart = x + scaled[:, half:]
    assert (scaled[:, half:] != 0).mean() > 0.9 and (apart.view(np.uint32) & 0xff != 0).mean() > 0.5
    np.testing.assert_array_equal(scaled[:, :half], apart)
