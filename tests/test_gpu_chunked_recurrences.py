"""The state layers' recurrences 16 rows at a time (stack_chunk.hip) against the float64 oracles, where the chunks can go wrong: portions that end
on, ahead of and behind a chunk's edge, state carried into and out of a chunked portion, steps of entries with very unequal row counts
(one row beside a hundred), every number of state tiles, columns that do not fill their group of 16, decays that vanish inside a
chunk and decays that are all but one."""
import numpy as np
import pytest

import narurax_cases
import rofozen_cases
import test_gpu_narurax
import test_gpu_rofozen
import test_gpu_tolenex
import tolenex_cases

pytestmark = pytest.mark.gpu


def hgrn2(dim, vdim, heads=2):
    return (test_gpu_tolenex, tolenex_cases.make_config([tolenex_cases.hgrn2_layer(heads=heads, dim=dim, vdim=vdim)]), 'mix.f.b')


def mamba2(dim, vdim, heads=4, groups=2):
    return (test_gpu_rofozen, rofozen_cases.make_config([rofozen_cases.mamba_layer(heads=heads, vdim=vdim, state=dim, groups=groups)]), 'mix.A_log')


def delta(dim, vdim, heads=4):
    return (test_gpu_narurax, narurax_cases.make_config([narurax_cases.delta_layer(heads=heads, kv_heads=2, dim=dim, vdim=vdim)]), 'mix.dt_bias')


KINDS = {'hgrn2': hgrn2, 'mamba2': mamba2, 'delta': delta}
RANGE = {'hgrn2': (-20.0, 20.0), 'mamba2': (-12.0, 4.0), 'delta': (-15.0, 12.0)}  # of the parameter that sets the decays: none left to all kept
SCHEDULES = {
    'whole': [[('a', 97)]],
    'edges': [[('a', 32)], [('a', 33)], [('a', 47)], [('a', 1)], [('a', 48)], [('a', 2)]],
    'unequal': [[('a', 1), ('b', 100), ('c', 16)], [('a', 64), ('b', 1), ('c', 17)], [('c', 31), ('a', 33), ('d', 32)], [('a', 1), ('b', 1), ('c', 1), ('d', 1)]],
}


def run(kind, dim, vdim, dtype, schedule, extreme=False):
    mod, cfg, decay = KINDS[kind](dim, vdim)
    steps = SCHEDULES[schedule]
    n = {}
    for step in steps:
        for rid, k in step:
            n[rid] = n.get(rid, 0) + k
    reqs = {rid: mod.tokens_for(cfg, k, 3 + i) for i, (rid, k) in enumerate(n.items())}
    w = mod.random_weights(cfg, 11)
    if extreme:
        a = w['l0.' + decay]
        lo, hi = RANGE[kind]
        w['l0.' + decay] = tolenex_cases.bf16_round(np.random.default_rng(5).uniform(lo, hi, a.shape).astype(np.float32))
        if kind == 'hgrn2':
            w['l0.mix.lower'] = np.zeros_like(w['l0.mix.lower'])
    got = mod.replay(mod.session_for(cfg, w, dtype), reqs, steps)
    for rid, toks in reqs.items():
        if kind == 'mamba2':
            mod.check(got[rid], mod.O.logits(toks, mod.as_f64(w), cfg), mod.tol_of(dtype), rid)
        else:
            mod.check_rows(got[rid], toks, w, cfg, dtype, rid)


@pytest.mark.parametrize('schedule', sorted(SCHEDULES))
@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('dim,vdim', [(64, 16), (128, 40), (192, 24), (256, 8)])
@pytest.mark.parametrize('kind', sorted(KINDS))
def test_portions(kind, dim, vdim, dtype, schedule):
    run(kind, dim, vdim, dtype, schedule)


@pytest.mark.parametrize('kind', sorted(KINDS))
def test_decays_from_none_to_all_in_one_chunk(kind):
    run(kind, 64, 24, 'float32', 'unequal', extreme=True)
