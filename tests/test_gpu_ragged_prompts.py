"""Prompts of unequal length, whose padding rows the context phase leaves out where that saves a row tile (tllm_session_context): against each prompt by itself, which has none -
batches just inside and outside of the rule, a prompt of one token among long ones, and a batch of the same session whose padding reaches into what an earlier one left.  Which of them
pack is what test_stack_host_runtime.py checks, without a GPU."""
import numpy as np
import pytest

from oracle import quant_oracle as QO
from tensorrt_llm.runtime.native import NativeSession
from test_gpu_session import synth_model

pytestmark = pytest.mark.gpu
S, NEW = 352, 4
BATCHES = [(352, 176, 240, 350), (352, 352, 352, 352), (352, 352, 352, 177), (352, 352, 352, 176), (352, 1, 352, 2), (1, 3, 1, 1)]  # 1408 rows, 11 x 48 tiles: up to 1232 pack


def sessions(mode, int8_kv):
    """-> prompts, and a function that sets up a session of such a model."""
    cfg, w = synth_model(51, L=2, H=16, D=2048, I=512)
    r = np.random.default_rng(19)
    ids = r.integers(3, cfg['vocab_size'], (4, S)).astype(np.int32)
    qmodel = QO.quantise_model(cfg, w, mode, int8_kv, calib_ids=ids[:, :40], calib_lens=np.full(4, 40, np.int32))

    def session(batch, prompt):
        s = NativeSession(dict(cfg, quant_mode=qmodel['quant_mode']))
        for k, v in qmodel['engine_tensors'].items():
            s.set_tensor(k, v)
        s.finalize()
        s.setup(batch, prompt, NEW)
        return s
    return ids, session


@pytest.mark.parametrize('mode,int8_kv', [('fp16', 0), ('fp16', 1), ('woq8', 1), ('sq_static_pc', 1)])
def test_a_ragged_batch_is_its_prompts(mode, int8_kv):
    ids, session = sessions(mode, int8_kv)

    def run(s, prompts, lens):
        s.context(prompts, np.array(lens, np.int32))
        first = s.logits()
        s.step(NEW - 1, use_graph=False)
        return first, s.logits(), s.output_ids()[:, -NEW:]

    alone, last_steps = {}, []
    many = session(4, S)
    for lens in BATCHES:
        padded = np.full((4, S), 2, np.int32)
        for b, n in enumerate(lens):
            padded[b, :n] = ids[b, :n]
        got = run(many, padded, lens)
        for b, n in enumerate(lens):
            if (b, n) not in alone:
                one = session(1, n)
                alone[b, n] = run(one, ids[b:b + 1, :n], (n, ))
                one.close()
            first, last, out = alone[b, n]
            # fp16 rounding of sums in another order (2^-11 a value, grown by the layers); the last step's only where the same tokens were chosen
            scale = max(np.abs(first).max(), 1.0)
            np.testing.assert_allclose(got[0][b], first[0], atol=2e-2 * scale, err_msg=f'{lens} prompt {b}')
            last_steps.append((got[2][b] == out[0]).all())
            if last_steps[-1]:
                np.testing.assert_allclose(got[1][b], last[0], atol=2e-2 * scale, err_msg=f'{lens} prompt {b}, last step')
    assert np.mean(last_steps) > 0.5
    many.close()
