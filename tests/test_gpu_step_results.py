"""What a step hands back (stack_ops.hip deliver_kernel, and the copies that take more rows): logits and greedy choices at vocabularies of one
part, of many, and of longer parts (from 64 x 2048 values), with ragged ends; rows on both sides of the line between the two ways;
equal logits (the lowest place), rows without a number, growing and shrinking numbers of rows on one engine."""
import numpy as np
import pytest

from rofozen_cases import make_config, mamba_layer, random_weights
from test_gpu_rofozen import O, as_f64, check, session_for, tol_of, tokens_for

pytestmark = pytest.mark.gpu


def run(vocab, rows, w_of=lambda w: w):
    cfg = make_config([mamba_layer()], width=40, vocab=vocab)
    w = w_of(random_weights(cfg, 3))
    s = session_for(cfg, w, 'float32')
    out = []
    for i, n in enumerate(rows):
        toks = tokens_for(cfg, n, 5 + i)
        logits, ids = s.step([(i, toks, list(range(n)))], end=(i,))
        out.append((toks, np.array(logits), np.array(ids)))
    return cfg, w, out


@pytest.mark.parametrize('vocab,rows', [(3, (1, 5)), (211, (1, 200, 7)), (2048, (1, 256, 2)), (2051, (3, 255, 256)), (16000, (131, 132, 1)), (131073, (1, 15, 16)),
                                        (200004, (1, 10, 11))])
def test_logits_and_choices(vocab, rows):
    cfg, w, out = run(vocab, rows)
    for toks, logits, ids in out:
        check(logits, O.logits(toks, as_f64(w), cfg), tol_of('float32'), len(toks))
        np.testing.assert_array_equal(ids, logits.argmax(-1))


@pytest.mark.parametrize('vocab', [211, 9000])
def test_equal_and_missing_numbers(vocab):
    def equal(w):  # rows v and vocab - 1 - v of the head are the same: every largest logit stands twice
        w['head'][vocab - vocab // 2:] = w['head'][:vocab // 2][::-1]
        return w

    def missing(w):
        w['head'][:] = np.nan
        return w
    for n in (1, 300):
        _, _, out = run(vocab, (n,), equal)
        np.testing.assert_array_equal(out[0][2], out[0][1].argmax(-1))
        assert (out[0][2] <= vocab // 2).all()
        _, _, out = run(vocab, (n,), missing)
        assert np.isnan(out[0][1]).all() and (out[0][2] == 0).all()
