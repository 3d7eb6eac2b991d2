"""Steps of one row per entry, where the recurrence's step kernel forms the convolution itself (stack_conv_impl.h) on a ring of raw inputs that prompts write as well:
sequences that begin with single tokens or with prompts of 1 .. 5, steps of single rows behind steps of several in between, a slot that an earlier sequence used,
channels that heads share and such that fill a workgroup's threads several times; positions that do not continue a sequence."""
import numpy as np
import pytest

import narurax_cases as N
import rofozen_cases as M
import test_gpu_narurax
import test_gpu_rofozen

pytestmark = pytest.mark.gpu

LAYERS = {'small': M.mamba_layer(heads=2, vdim=4, state=8, groups=1), 'shared': M.mamba_layer(heads=6, vdim=12, state=16, groups=2),
          'plain': M.mamba_layer(heads=4, vdim=64, state=128, groups=4), 'long': M.mamba_layer(heads=2, vdim=4, state=1024, groups=1),
          'delta small': N.delta_layer(heads=2, kv_heads=1, dim=8, vdim=4), 'delta shared': N.delta_layer(heads=6, kv_heads=2, dim=16, vdim=12),
          'delta plain': N.delta_layer(heads=2, kv_heads=2, dim=128, vdim=128), 'delta wide': N.delta_layer(heads=1, kv_heads=1, dim=8, vdim=512)}
FIRST = [{'a': 19, 'b': 12}, {'c': 3, 'd': 7, 'e': 9}, {'f': 2, 'g': 14}]
# first of each: rows of every request's first step, by the requests' order; later ones: single rows, and some of several
STARTS = [(1, 1), (2, 5, 3), (1, 4)]


def schedule(reqs, starts):
    left = dict(reqs)
    steps = []
    while any(left.values()):
        step = []
        for (name, n), first in zip(reqs.items(), starts):
            rows = min(left[name], first if left[name] == n else 3 if len(steps) == 6 else 1)
            if rows:
                step.append((name, rows))
                left[name] -= rows
        steps.append(step)
    return steps


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('layer', sorted(LAYERS))
def test_steps_of_single_rows(layer, dtype):
    cases, test = (N, test_gpu_narurax) if layer.startswith('delta') else (M, test_gpu_rofozen)
    cfg = cases.make_config([LAYERS[layer], LAYERS[layer]])
    w = test.weights_for(cfg, 5, dtype)
    s = test.session_for(cfg, w, dtype, max_sequences=3)
    for i, (reqs, starts) in enumerate(zip(FIRST, STARTS)):
        toks = {name: test.tokens_for(cfg, n, 10 * i + n) for name, n in reqs.items()}
        got = test.replay(s, toks, schedule(reqs, starts))
        for name in toks:
            test.check_rows(got[name], toks[name], w, cfg, dtype, f'{layer} {name}')


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('taps', [3, 4])
@pytest.mark.parametrize('layer', ['shared', 'delta shared'])
def test_positions_that_do_not_continue(layer, taps, dtype):
    """The convolution's history is what the sequence was fed last, whatever positions its caller counts: the same bits as with positions that continue."""
    cases, test = (N, test_gpu_narurax) if layer.startswith('delta') else (M, test_gpu_rofozen)
    kind = dict(LAYERS[layer], mixer=dict(LAYERS[layer]['mixer'], conv=taps))
    cfg = cases.make_config([kind, kind])
    w = test.weights_for(cfg, 5, dtype)
    toks, rows = test.tokens_for(cfg, 24, 6), (5, 1, 1, 1, 3, 1, 1, 1, 2, 6, 1, 1)
    got = []
    for places in (None, (0, 9, 9, 9, 4, 5, 30, 31, 1, 2, 1, 8)):
        e = test.session_for(cfg, w, dtype, max_sequences=2).engine
        out, at = [], 0
        for k, n in enumerate(rows):
            out.append(e.step(toks[at:at + n], [n], [places[k] if places else at], [1], [[0]], list(range(n)))[0])
            at += n
        got.append(np.concatenate(out))
    np.testing.assert_array_equal(*got)
