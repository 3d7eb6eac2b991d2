"""LLaMA decode attention of sequences within one split (mmha_decode.hip), which finish their row in the launch without partials, and what follows it:
generation across the slot at which a second split begins (192 at head size 128: partials, tickets, the merge in the launch) and cache lengths on
both sides of the short form's (64)."""
import numpy as np
import pytest

from oracle import quant_oracle as QO
from tensorrt_llm.runtime.native import NativeSession
from test_gpu_session import synth_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('new', [4, 300], ids=['short form', 'long form'])
def test_a_head_whose_scores_are_no_numbers_counts_nothing(new):
    """A token whose query overflows in one head (infinities, and behind the rotation no numbers): no key has a share, and the head's row is zero,
    as the merge of such partials has it.  The oracle is the model whose O projection does not read that head; equal bits, since both add zeros."""
    cfg, w = synth_model(23, L=1, H=4, D=256, I=512, V=128)
    w = {k: v.copy() for k, v in w.items()}
    token, dim, head = 7, 100, 64
    w['vocab_embedding.weight'][:, dim] = 0
    w['vocab_embedding.weight'][token, dim] = 10
    r = np.random.default_rng(3)
    ids = r.integers(10, 128, (2, 12)).astype(np.int32)
    lens = np.array([12, 5], np.int32)
    ids[1, 5:] = 2
    runs = []
    for overflows in (True, False):
        x = {k: v.copy() for k, v in w.items()}
        x['layers.0.attention.qkv.weight'][:head, dim] = 6e4 if overflows else 0
        if not overflows:
            x['layers.0.attention.dense.weight'][:, :head] = 0
        s = NativeSession(dict(cfg, quant_mode=0))
        for k, v in x.items():
            s.set_tensor(k, v)
        s.finalize()
        s.setup(2, 12, new)
        s.context(ids, lens)
        logits = []
        for graph in (False, True, True):
            s.force_tokens(np.full(2, token, np.int32))
            s.step(1, use_graph=graph)
            logits.append(s.logits().copy())
        s.close()
        runs.append(np.stack(logits))
    for logits in runs:
        assert not np.isnan(logits).any()
    np.testing.assert_array_equal(runs[0], runs[1])


@pytest.mark.parametrize('prompt,new', [(187, 10), (54, 10), (55, 10)], ids=['across slot 192', '64 slots', '65 slots'])
@pytest.mark.parametrize('mode,int8_kv', [('fp16', 0), ('sq_static_pc', 1)])
def test_generation_vs_oracle(mode, int8_kv, prompt, new):
    """Every step, eager and captured, in a ragged batch.  fp16: the logits, bounds of test_gpu_session's test_quantised_paths_vs_oracle.  SmoothQuant: the
    int8 rows that the first layer's attention launch leaves for the O projection, at most one step from the oracle's and a quarter of them off, as in
    test_gpu_session's test_sq_int8_taps_at_all_four_quantisers_in_lsbs (a flipped integer grows from layer to layer, and logits say little)."""
    cfg, w = synth_model(31, L=2, H=2, D=256, I=512, V=512)
    r = np.random.default_rng(8)
    ids = r.integers(3, cfg['vocab_size'], (2, prompt)).astype(np.int32)
    lens = np.array([prompt, prompt - 30], np.int32)
    ids[1, lens[1]:] = 2
    qmodel = QO.quantise_model(cfg, w, mode, int8_kv, calib_ids=ids, calib_lens=lens)
    s = NativeSession(dict(cfg, quant_mode=qmodel['quant_mode'], debug_taps=int(mode != 'fp16')))
    for k, v in qmodel['engine_tensors'].items():
        s.set_tensor(k, v)
    s.finalize()
    s.setup(2, prompt, new)
    runs = []
    for graph in (False, True):
        s.context(ids, lens)
        logits, rows = [s.logits().copy()], []
        for _ in range(new - 1):
            s.step(1, use_graph=graph)
            logits.append(s.logits().copy())
            if mode != 'fp16':
                rows.append(s.tap(0, 'o_in', 256, quantised=True))
        runs.append((logits, rows, s.output_ids()))
    s.close()
    (logits, rows, out), captured = runs
    for a, b in zip(runs[0], captured):
        np.testing.assert_array_equal(np.array(a), np.array(b))
    taps = {}
    ref, _ = QO.run_model(qmodel, ids, lens, new, feed_ids=out[:, prompt:prompt + new], taps=taps)
    if mode == 'fp16':
        scale = max(np.abs(ref[0]).max(), 1.0)
        for g, x in zip(logits, ref):
            np.testing.assert_allclose(g, x, atol=1e-2 * scale)
            assert np.abs(g - x).mean() < 2.5e-3 * scale
    for g, x in zip(rows, taps['gemm_in']):
        d = np.abs(g.astype(np.int32) - x[0]['o_in'].astype(np.int32))
        assert d.max() <= 1 and (d != 0).mean() <= 0.25, (d.max(), (d != 0).mean())
