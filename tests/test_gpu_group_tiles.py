"""Grouped bfloat16 products whose groups fit one 256-row tile (launch_glds_bf16 of stack_gemm.hip takes 256 x 256 tiles where that saves a round of
workgroups: 8 groups of 200 rows on average x 8176 columns on 256 CUs): groups that end inside the tile, columns that end inside it, one stage of K and
several.  Bounds as in test_gpu_product_tiles."""
import pytest

import ruzinex_cases as Z
import sodudra_cases
import test_gpu_ruzinex as R
import test_gpu_sodudra as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('rows', [752, 800])
@pytest.mark.parametrize('k', [64, 320])
def test_groups_of_one_wide_tile(k, rows):
    cfg = Z.make_config([Z.layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=Z.moe(experts=8, top=2, ff=4088, shared=0))], width=k)
    toks = R.tokens_for(cfg, rows, 97)
    w = R.weights_for(cfg, 98, 'bfloat16', toks)
    R.check_rows(R.replay(R.session_for(cfg, w, 'bfloat16'), {'a': toks}, [[('a', rows)]])['a'], toks, w, cfg, 'bfloat16')


# Every group has all of a step's rows, or what two choices of each leave it: on both sides of the heights that a tile of up to 288 rows x 192 columns comes in (steps of 32 rows, two
# tiles from 289 on), columns that end inside a tile (5888 = 30.7 of them; the down product's 512 and 576 = 2.7 and 3), eight K-tiles and nine.
@pytest.mark.parametrize('k', [512, 576])
@pytest.mark.parametrize('rows,top', [(72, 8), (90, 8), (97, 8), (129, 8), (161, 8), (200, 8), (225, 8), (257, 8), (288, 8), (289, 8), (330, 8), (760, 2), (1000, 2)])
def test_groups_of_tall_tiles(rows, top, k):
    cfg = Z.make_config([Z.layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=Z.moe(experts=8, top=top, ff=2944, shared=0))], width=k)
    toks = R.tokens_for(cfg, rows, 97)
    w = R.weights_for(cfg, 98, 'bfloat16', toks)
    R.check_rows(R.replay(R.session_for(cfg, w, 'bfloat16'), {'a': toks}, [[('a', rows)]])['a'], toks, w, cfg, 'bfloat16')


# Experts without a gate (squared ReLU), whose results leave as they are: heights of one to nine steps, one tile and two, columns that end inside a tile (5888 = 30.7 of them).
UNGATED_ROWS = (40, 72, 129, 161, 200, 257, 288, 289, 330)


def ungated_config(cases):
    return cases.make_config([cases.layer(heads=2, dim=16, vdim=16, kv_rank=32, mlp=cases.moe(experts=8, top=8, ff=5888, shared=0))], width=512, side=0)


@pytest.mark.parametrize('rows', UNGATED_ROWS)
def test_tall_tiles_of_ungated_experts(rows):
    cfg = ungated_config(sodudra_cases)
    toks = S.tokens_for(cfg, rows, 97)
    w = S.weights_for(cfg, 98, 'bfloat16', toks)
    S.check_rows(S.replay(S.session_for(cfg, w, 'bfloat16'), {'a': toks}, [[('a', rows)]])['a'], toks, w, cfg, 'bfloat16')
