"""Products of 2 .. 31 rows in every launch shape of the weight-streaming form (pick_shape of gemm_slim_impl.h): on both sides of its lines in rows
(8, 16), columns (2048, 4096, 12288, 16384 on 256 CUs) and length of a row (512, 1024, 4096 bytes), with columns that end inside a workgroup and rows that end inside a
block, in its second run, or give some waves no block.  The stack engine's against exactly known rows; bounds of the plugins as in
test_gpu_few_rows."""
import numpy as np
import pytest
import torch

import ruzinex_cases as Z
import test_gpu_ruzinex as R
from helpers import as_f32, f32, i32, make_plugin, run_plugin
from oracle import llama_oracle as O
from tensorrt_llm.plugin import capi

pytestmark = pytest.mark.gpu

ROWS = [2, 8, 9, 16, 17, 31]
COLUMNS = [2045, 3003, 4101]


def known_rows(n, k, m, **kw):
    """A session, a prompt of m tokens and the bfloat16 rows h that its head multiplies, known exactly: the layer adds nothing to embeddings of +- 1,
    whose norm is 1 / sqrt(1 + eps), 5e-6 below 1, and takes every bfloat16 weight back to itself."""
    cfg = Z.make_config([Z.layer(heads=2, kv_heads=1, dim=32, vdim=32)], width=k, vocab=n)
    w = Z.random_weights(cfg, 6)
    w['l0.mix.o'][:] = 0
    signs = np.random.default_rng(5).integers(0, 2, (m, k)) * 2.0 - 1
    w['embed'][:m] = signs
    return R.session_for(cfg, w, 'bfloat16', debug_mode=True, **kw), list(range(m)), signs * w['final.norm'], w['embed'].astype(np.float64)


def check_head(got, h, w):
    """Sums of k products that are exact in fp32: each is off by no more than k roundings of what its terms come to."""
    worst = np.abs(got - h @ w.T) / (np.abs(h) @ np.abs(w).T)
    assert (worst < h.shape[1] * 2.0 ** -24).all(), f'place {np.unravel_index(worst.argmax(), worst.shape)} is off by {worst.max():.3g} of its terms'


@pytest.mark.parametrize('k', [8, 136, 264, 2048, 2056, 4360])
@pytest.mark.parametrize('n', COLUMNS)
@pytest.mark.parametrize('m', ROWS)
def test_stack_products(m, n, k):
    s, toks, h, w = known_rows(n, k, m)
    got, _ = s.step([('a', toks, list(range(m)))])
    np.testing.assert_array_equal(s.engine.tap(0), w[:m])
    check_head(got, h, w)


@pytest.mark.parametrize('k', [8, 72, 264, 520, 1544, 2040, 2048, 2056])
@pytest.mark.parametrize('n', [12301, 16371])
def test_stack_products_of_many_columns(n, k):
    """More than three, and four, workgroups of 16 columns per CU."""
    s, toks, h, w = known_rows(n, k, max(ROWS), max_sequences=len(ROWS))
    for m in ROWS:
        got, _ = s.step([(m, toks[:m], list(range(m)))])
        check_head(got, h[:m], w)


@pytest.mark.parametrize('k', [64, 544, 4112, 8208])
@pytest.mark.parametrize('n', COLUMNS)
@pytest.mark.parametrize('m', [5, 8, 9, 17])
@pytest.mark.parametrize('kind', ['fp16', 'sq'])
def test_llama_products(kind, m, n, k):
    r = np.random.default_rng(m * 7919 + n)
    out = torch.empty((m, n), dtype=torch.float16, device='cuda')
    if kind == 'sq':  # exact
        a, w = [torch.from_numpy(r.integers(-128, 128, s).astype(np.int8)) for s in ((m, k), (n, k))]
        sa, sb = [torch.from_numpy(r.uniform(0.001, 0.01, s).astype(np.float32)) for s in ((m, 1), (1, n))]
        p = make_plugin('SmoothQuantGemm', [('has_per_channel_scaling', i32(1)), ('has_per_token_scaling', i32(1)), ('type_id', i32([capi.HALF]))])
        run_plugin(p, [a.cuda(), w.cuda(), sa.cuda(), sb.cuda()], [out])
        np.testing.assert_array_equal(as_f32(out), O.sq_gemm(a.numpy(), w.numpy(), sa.numpy(), sb.numpy(), 'float16'))
        return
    x = r.standard_normal((m, k)).astype(np.float16)
    w = (r.standard_normal((n, k)) / np.sqrt(k)).astype(np.float16)
    p = make_plugin('Gemm', [('transa', i32(0)), ('transb', i32(1)), ('type_id', i32([capi.HALF]))])
    run_plugin(p, [torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda()], [out])
    want = x.astype(np.float64) @ w.astype(np.float64).T
    mags = np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T
    assert (np.abs(as_f32(out) - want) <= 2.0 ** -10 * np.abs(want) + (k * 2.0 ** -24 + 2.0 ** -16) * mags).all()
