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


def check_request(mod, kind, got, toks, w, cfg, dtype, rid):
    if kind == 'mamba2':
        mod.check(got, mod.O.logits(toks, mod.as_f64(w), cfg), mod.tol_of(dtype), rid)
    else:
        mod.check_rows(got, toks, w, cfg, dtype, rid)


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
        check_request(mod, kind, got[rid], toks, w, cfg, dtype, rid)


@pytest.mark.parametrize('schedule', sorted(SCHEDULES))
@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('dim,vdim', [(64, 16), (128, 40), (192, 24), (256, 8)])
@pytest.mark.parametrize('kind', sorted(KINDS))
def test_portions(kind, dim, vdim, dtype, schedule):
    run(kind, dim, vdim, dtype, schedule)


@pytest.mark.parametrize('kind', sorted(KINDS))
def test_decays_from_none_to_all_in_one_chunk(kind):
    run(kind, 64, 24, 'float32', 'unequal', extreme=True)


@pytest.mark.parametrize('where', [33, 47, 96])
@pytest.mark.parametrize('what', ['row', 'value'])
@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('kind', sorted(KINDS))
def test_a_row_without_finite_numbers_leaves_the_earlier_ones_alone(kind, dtype, what, where):
    """Row `where` of a request is NaN in every channel, or its values overflow: the rows before it, in the same chunk too, are what the oracle
    has for the prompt that ends there, and the request beside it is untouched.  (The last place is a chunk of one row.)"""
    bad_row(kind, dtype, what, where, 64, 24, 97)


def bad_row(kind, dtype, what, where, dim, vdim, rows):
    mod, cfg, _ = KINDS[kind](dim, vdim)
    toks, other = mod.tokens_for(cfg, rows, 3), mod.tokens_for(cfg, 20, 4)
    bad = next(t for t in range(cfg['vocab']) if t not in toks and t not in other)
    w = mod.random_weights(cfg, 11)
    if what == 'row':
        w['embed'][bad] = np.nan
    else:  # channel 0 is the bad token's alone, and the values read it with a weight near the type's largest
        for name in ('embed', 'bigram'):
            if name in w:
                w[name][:, 0] = 0.0
        w['embed'][bad, 0] = 20.0
        w['l0.norm1'][0] = 1.0
        if kind == 'mamba2':
            inner = 4 * vdim
            w['l0.mix.in'][inner:2 * inner, 0] = tolenex_cases.bf16_round(np.float32(3e38))
        else:
            w['l0.mix.v'][:, 0] = tolenex_cases.bf16_round(np.float32(3e38))
    toks[where] = bad
    got = mod.replay(mod.session_for(cfg, w, dtype), {'b': other, 'a': toks}, [[('b', 20), ('a', rows)]])
    assert not np.isfinite(got['a'][where]).all()
    check_request(mod, kind, got['a'][:where], toks[:where], w, cfg, dtype, 'a')
    check_request(mod, kind, got['b'], other, w, cfg, dtype, 'b')


# Portions of 112 .. 257 rows: around eight chunks, one that begins with carried state (which walk a step of them has: test_stack_host_runtime.py).
@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('dim,vdim', [(64, 24), (128, 16)])
@pytest.mark.parametrize('kind', ['hgrn2', 'mamba2'])
def test_portions_around_eight_chunks(kind, dim, vdim, dtype, monkeypatch):
    monkeypatch.setitem(SCHEDULES, 'eights', [[('a', 112), ('b', 128)], [('a', 129), ('b', 32)], [('a', 127), ('b', 257)], [('a', 144), ('b', 1)]])
    run(kind, dim, vdim, dtype, 'eights')


# The walk of eight chunks between two barriers: full turns and one short of them, entries beside the longest that end in, on and behind a turn or have a single row, carried state; 64 rows
# of state from 46 chunks (Mamba-2: 24) on.
@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('dim,vdim', [(64, 24), (128, 16)])
@pytest.mark.parametrize('kind', ['hgrn2', 'mamba2'])
def test_turns_of_eight_chunks(kind, dim, vdim, dtype, monkeypatch):
    steps = EIGHT_CHUNKS[dim]
    monkeypatch.setitem(SCHEDULES, 'turns', steps)
    run(kind, dim, vdim, dtype, 'turns')


EIGHT_CHUNKS = {128: [[('a', 128), ('b', 113)], [('a', 129), ('b', 241), ('c', 1)], [('a', 1), ('b', 16), ('c', 313)]], 64: [[('a', 40)], [('a', 752), ('b', 129)]]}


@pytest.mark.parametrize('where', [33, 47, 112])
@pytest.mark.parametrize('what', ['row', 'value'])
@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('kind', ['hgrn2', 'mamba2'])
def test_a_row_without_finite_numbers_in_a_turn_of_eight_chunks(kind, dtype, what, where):
    bad_row(kind, dtype, what, where, 128, 16, 113)
