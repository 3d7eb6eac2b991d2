"""LLaMA decode attention of sequences within one split (mmha_decode.hip), which finish their row in the launch without partials."""
import numpy as np
import pytest

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
