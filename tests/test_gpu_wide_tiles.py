"""The 256 x 256 tiles of gemm_wide_impl.h in a step: K-tiles in every position of the operands' rings (three buffers, two), a last row tile of more and of
less than 128 rows, columns that end inside a tile, several rounds of tiles, every way out (16-bit and fp32 rows, gated pairs, the fp32 residual with and
without a gate), groups, more than 64 of them too.  That these sizes take them is what test_stack_host_runtime.py checks, without a GPU."""
import pytest

import ruzinex_cases as Z
import sodudra_cases as S
import test_gpu_product_tiles as P
import test_gpu_ruzinex as R
import test_gpu_sodudra
import test_gpu_tolenex
import tolenex_cases as T

pytestmark = pytest.mark.gpu

PLAIN = [(rows, k) for rows in (1000, 800) for k in (2496, 2560, 2624)]
COLUMNS = 16008
GATED = (800, 2496, 8000)                                       # rows, width, ff
GROUPED = [(1000, 1088, 2, 2, 4032), (1000, 1152, 2, 2, 4032), (1000, 320, 80, 32, 192)]  # tokens, width, experts, choices, ff
RESIDUAL = (4096, 4096, 2496)                                   # rows, width, K of the product


def gated_config():
    return P.gated_config(Z.dense(ff=GATED[2]), GATED[1])


def grouped_config(width, experts, top, ff):
    return P.gated_config(Z.moe(experts=experts, top=top, ff=ff, shared=0), width)


def residual_config(cases):
    width, ff = RESIDUAL[1:]
    if cases is T:
        return T.make_config([T.attention_layer(heads=4, kv_heads=1, dim=32, vdim=64, rot_dims=16, ff=ff)], width=width, groups=2)
    return S.make_config([S.layer(heads=4, dim=32, vdim=32, kv_rank=64, mlp=S.moe(experts=2, top=1, ff=32, shared=ff - 4 * 32))], width=width, side=0)


@pytest.mark.parametrize('rows,k', PLAIN)
def test_plain_product(rows, k, monkeypatch):
    monkeypatch.setattr(P, 'ROWS', rows)
    P.plain(COLUMNS, k)


def test_gated_product():
    cfg = gated_config()
    toks = R.tokens_for(cfg, GATED[0], 97)
    w = Z.random_weights(cfg, 98)
    R.check_rows(R.replay(R.session_for(cfg, w, 'bfloat16'), {'a': toks}, [[('a', GATED[0])]])['a'], toks, w, cfg, 'bfloat16')


@pytest.mark.parametrize('tokens,width,experts,top,ff', GROUPED)
def test_grouped_product(tokens, width, experts, top, ff):
    cfg = grouped_config(width, experts, top, ff)
    toks = R.tokens_for(cfg, tokens, 97)
    w = R.weights_for(cfg, 98, 'bfloat16', toks)
    R.check_rows(R.replay(R.session_for(cfg, w, 'bfloat16'), {'a': toks}, [[('a', tokens)]])['a'], toks, w, cfg, 'bfloat16')


def test_gated_residual():
    cfg = residual_config(T)
    toks = test_gpu_tolenex.tokens_for(cfg, RESIDUAL[0], 5)
    w = T.random_weights(cfg, 6)
    s = test_gpu_tolenex.session_for(cfg, w, 'bfloat16', max_tokens=RESIDUAL[0], max_batch_tokens=RESIDUAL[0])
    test_gpu_tolenex.check_rows(T.replay(s, {'a': toks}, [[('a', RESIDUAL[0])]])['a'], toks, w, cfg, 'bfloat16')


def test_residual():
    """The mixer's heads and the shared feed-forward land in one product."""
    cfg = residual_config(S)
    toks = test_gpu_sodudra.tokens_for(cfg, RESIDUAL[0], 5)
    w = S.random_weights(cfg, 6)
    s = test_gpu_sodudra.session_for(cfg, w, 'bfloat16', max_tokens=RESIDUAL[0], max_batch_tokens=RESIDUAL[0])
    test_gpu_sodudra.check_rows(T.replay(s, {'a': toks}, [[('a', RESIDUAL[0])]])['a'], toks, w, cfg, 'bfloat16')
