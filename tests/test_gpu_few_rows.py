"""Products of few rows (2 .. 31; LLaMA: from 5, int4 weights and fp16 O / down of a generation step from 3) through the weight-streaming MFMA kernels
(gemm_slim_impl.h): LLaMA plugins in every weight type and the stack engine, at the edges of the row tiles (9, 16, 17, 31 rows), ragged columns, rows
of W that end inside a 256-byte block or are shorter than the waves' first round.  Weight-only weights: both launch shapes (from 5120 columns on);
the launch shapes of the others are test_gpu_slim_shapes.py's."""
import numpy as np
import pytest
import torch

from helpers import as_f32, f32, h, i32, make_plugin, run_plugin
from oracle import llama_oracle as O
from tensorrt_llm.plugin import capi

pytestmark = pytest.mark.gpu

SHAPES = [(3, 64, 1184), (5, 40, 320), (8, 1003, 2080), (9, 13, 64), (16, 40, 320), (17, 272, 1184), (31, 1003, 2080), (24, 64, 4096), (31, 5136, 544), (12, 5121, 256)]


@pytest.mark.parametrize('m,n,k', SHAPES)
@pytest.mark.parametrize('kind', ['fp16', 'sq', 'woq8', 'woq4'])
def test_llama_products_of_few_rows(kind, m, n, k):
    r = np.random.default_rng(m * 7919 + n)
    out = torch.empty((m, n), dtype=torch.float16, device='cuda')
    if kind == 'sq':  # exact
        a, w = [torch.from_numpy(r.integers(-128, 128, s).astype(np.int8)) for s in ((m, k), (n, k))]
        sa, sb = [torch.from_numpy(r.uniform(0.01, 0.1, s).astype(np.float32)) for s in ((m, 1), (1, n))]
        p = make_plugin('SmoothQuantGemm', [('has_per_channel_scaling', i32(1)), ('has_per_token_scaling', i32(1)), ('type_id', i32([capi.HALF]))])
        run_plugin(p, [a.cuda(), w.cuda(), sa.cuda(), sb.cuda()], [out])
        np.testing.assert_array_equal(as_f32(out), O.sq_gemm(a.numpy(), w.numpy(), sa.numpy(), sb.numpy(), 'float16'))
        return
    x = r.standard_normal((m, k)).astype(np.float16)
    w = (r.standard_normal((k, n)) / np.sqrt(k)).astype(np.float16)
    if kind == 'fp16':
        p = make_plugin('Gemm', [('transa', i32(0)), ('transb', i32(1)), ('type_id', i32([capi.HALF]))])
        run_plugin(p, [torch.from_numpy(x).cuda(), torch.from_numpy(np.ascontiguousarray(w.T)).cuda()], [out])
        want = x.astype(np.float64) @ w.astype(np.float64)
    else:
        bits = 8 if kind == 'woq8' else 4
        if n % (4 if bits == 8 else 8):
            pytest.skip('the quantiser packs whole 32-bit words of columns')
        q, scales, _ = capi.symmetric_quantize_last_axis(w, bits)
        q_ref, s_ref = O.woq_quantize(w.astype(np.float32), bits)
        p = make_plugin('WeightOnlyQuantMatmul', [('type_id', i32([capi.HALF])), ('weight_type_id', i32(1 if bits == 8 else 2))])
        run_plugin(p, [torch.from_numpy(x).cuda(), torch.from_numpy(q).cuda().view(torch.float32).reshape(k, -1), torch.from_numpy(scales).cuda()], [out])
        want = (x.astype(np.float64) @ q_ref.astype(np.float64)) * s_ref.astype(np.float64)
    # k products exact, fp32 sums of k terms (k 2^-24 of the sum of magnitudes at the worst), one rounding to fp16 (2^-11)
    mags = np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64)
    assert (np.abs(as_f32(out) - want) <= 2.0 ** -10 * np.abs(want) + (k * 2.0 ** -24 + 2.0 ** -16) * mags).all()


@pytest.mark.parametrize('rows', [2, 5, 9, 16, 17, 31])
@pytest.mark.parametrize('model', ['tiled', 'odd', 'wide'])
def test_stack_products_of_few_rows(model, rows):
    """A prompt of `rows` tokens (every product has that many rows, every expert up to that many), then single tokens of it."""
    from ruzinex_cases import dense, layer, make_config, moe
    from test_gpu_ruzinex import TILED, check_rows, replay, session_for, tokens_for, weights_for
    cfg = {'tiled': TILED,
           'odd': make_config([layer(heads=3, kv_heads=1, dim=16, vdim=24, mlp=moe(experts=70, top=3, ff=40, shared=24)), layer(heads=3, kv_heads=1, dim=16, vdim=24, mlp=dense(ff=88))], width=136, vocab=203),
           'wide': make_config([layer(mlp=dense(ff=2600))], width=264, vocab=5127)}[model]
    toks = tokens_for(cfg, rows + 3, 5)
    w = weights_for(cfg, 31, 'bfloat16', toks)
    got = replay(session_for(cfg, w, 'bfloat16'), {'a': toks}, [[('a', rows)]] + [[('a', 1)]] * 3)['a']
    check_rows(got, toks, w, cfg, 'bfloat16')


@pytest.mark.parametrize('requests', [1, 3, 12, 30])
def test_stack_decode_of_many_requests(requests):
    """One token of each of `requests` requests per step: more experts than rows and the other way round."""
    from ruzinex_cases import dense, layer, make_config, moe
    from test_gpu_ruzinex import check_rows, replay, session_for, tokens_for, weights_for
    cfg = make_config([layer(heads=4, kv_heads=2, dim=32, vdim=32, rot_dims=32, mlp=moe(experts=70, top=2, ff=64, shared=64)),
                       layer(heads=4, kv_heads=2, dim=32, vdim=32, rot_dims=32, mlp=dense(ff=192))], width=128, vocab=211)
    reqs = {i: tokens_for(cfg, 4 + i % 3, 40 + i) for i in range(requests)}
    w = weights_for(cfg, 3, 'bfloat16', reqs)
    schedule = [[(i, 1 + i % 3)] for i in reqs] + [[(i, 1) for i in reqs]] * 3
    got = replay(session_for(cfg, w, 'bfloat16', max_tokens=64 * requests, max_sequences=requests), reqs, schedule)
    for i, toks in reqs.items():
        check_rows(got[i], toks, w, cfg, 'bfloat16', i)


@pytest.mark.parametrize('mode,int8_kv', [('fp16', 0), ('woq8', 1), ('woq4', 0)])
@pytest.mark.parametrize('batch', [2, 3, 5, 8, 17, 32, 33])
def test_llama_decode_of_several_sequences(batch, mode, int8_kv):
    """Generation steps whose products take the norm ahead of them and the residual or SwiGLU behind them, on both sides of the rows where
    that form starts and ends, eager and captured; bounds of test_gpu_session.test_quantised_paths_vs_oracle."""
    from oracle import quant_oracle as QO
    from tensorrt_llm.runtime.native import NativeSession
    from test_gpu_session import synth_model
    cfg, w = synth_model(11)
    S, NEW = 6, 4
    r = np.random.default_rng(batch)
    ids = r.integers(3, cfg['vocab_size'], (batch, S)).astype(np.int32)
    lens = r.integers(2, S + 1, batch).astype(np.int32)
    lens[0] = S
    for b in range(batch):
        ids[b, lens[b]:] = 2
    q = QO.quantise_model(cfg, w, mode, int8_kv, calib_ids=ids, calib_lens=lens)
    s = NativeSession(dict(cfg, quant_mode=q['quant_mode']))
    for k, v in q['engine_tensors'].items():
        s.set_tensor(k, v)
    s.finalize()
    s.setup(batch, S, NEW)
    s.context(ids, lens)
    got = [s.logits()]
    s.step(1, use_graph=False)
    got.append(s.logits())
    s.step(2, use_graph=True)
    got.append(s.logits())
    out = s.output_ids()
    s.close()
    ref, _ = QO.run_model(q, ids, lens, NEW, feed_ids=out[:, S:S + NEW])
    scale = max(np.abs(ref[0]).max(), 1.0)
    for g, want in ((got[0], ref[0]), (got[1], ref[1]), (got[2], ref[3])):
        np.testing.assert_allclose(g, want, atol=1e-2 * scale)
        assert np.abs(g - want).mean() < 2.5e-3 * scale
