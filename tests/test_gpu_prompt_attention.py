"""Attention over prompts (attn_prompt_kernel of stack_attn.hip) against the float64 oracles: every score and mask option over the 64-key units'
edges, in its three forms (few workgroups: waves share a unit's keys; more; many: two row tiles per wave), over portions that start inside a unit,
and over pages of 32 (the form before it), 64 and 128 keys.  bfloat16 engine, bounds of the designs' own tests."""
import numpy as np
import pytest

import narurax_cases
import ruzinex_cases
import test_gpu_narurax
import test_gpu_ruzinex
import test_gpu_tolenex
import test_gpu_vetipel
import tolenex_cases
import vetipel_cases
from tolenex_cases import as_f64

pytestmark = pytest.mark.gpu


def tolenex(heads, kv_heads, dim, vdim):
    return test_gpu_tolenex, tolenex_cases.make_config([tolenex_cases.attention_layer(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, rot_dims=32, ff=0)])


def ruzinex(heads, kv_heads, dim, vdim):
    return test_gpu_ruzinex, ruzinex_cases.make_config([ruzinex_cases.layer(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, rot_dims=32)])


def window(heads, kv_heads, dim, vdim):  # sigmoid weights, distance penalties, a window of 70
    return test_gpu_vetipel, vetipel_cases.make_config([vetipel_cases.window_layer(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, size=70, ff=0)])


def chunk(heads, kv_heads, dim, vdim):  # temperatures, logarithmic penalties, chunks of 90
    return test_gpu_vetipel, vetipel_cases.make_config([vetipel_cases.chunk_layer(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, size=90, ff=0)])


def kept(heads, kv_heads, dim, vdim):  # a window of 65 behind 5 kept keys
    return test_gpu_narurax, narurax_cases.make_config([narurax_cases.attn2_layer(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, rot_dims=32, size=65, keep=5)])


def talking(heads, kv_heads, dim, vdim):  # head-mixed weights: every head's weights over every value head's rows
    return test_gpu_narurax, narurax_cases.make_config([narurax_cases.attn_layer(heads=heads, kv_heads=kv_heads, dim=dim, rot_dims=32, size=130, keep=70)])


KINDS = {f.__name__: f for f in (tolenex, ruzinex, window, chunk, kept, talking)}
SCHEDULES = {'whole': [[('a', 193)]], 'portions': [[('a', 33)], [('a', 95)], [('a', 32), ('b', 65)], [('a', 64), ('b', 70)]]}


def run(kind, heads, kv_heads, dim, vdim, steps, page=64):
    mod, cfg = KINDS[kind](heads, kv_heads, dim, vdim)
    n = {}
    for step in steps:
        for rid, k in step:
            n[rid] = n.get(rid, 0) + k
    reqs = {rid: mod.tokens_for(cfg, k, 3 + i) for i, (rid, k) in enumerate(n.items())}
    w = mod.random_weights(cfg, 13)
    if page == 64:
        s = mod.session_for(cfg, w, 'bfloat16', max_tokens=2048)
    else:
        from tensorrt_llm.runtime import RaggedGenerationSession
        model = mod.as_model(cfg, w)
        model.page_size, plain = page, model.config.engine_config
        model.config.engine_config = lambda: dict(plain(), page_size=page)
        s = RaggedGenerationSession(model, dtype='bfloat16', max_tokens=2048, max_sequences=4)
    got = mod.replay(s, reqs, steps)
    for rid, toks in reqs.items():
        if mod is test_gpu_vetipel:
            mod.check(got[rid], mod.O.logits(toks, as_f64(w), cfg), mod.tol_of('bfloat16'), rid)
        else:
            mod.check_rows(got[rid], toks, w, cfg, 'bfloat16', rid)


@pytest.mark.parametrize('schedule', sorted(SCHEDULES))
@pytest.mark.parametrize('dim,vdim', [(64, 64), (128, 128), (192, 64), (64, 128)])
@pytest.mark.parametrize('kind', sorted(KINDS))
def test_every_option(kind, dim, vdim, schedule):
    if kind == 'tolenex' and dim == 192:
        pytest.skip('two maps of 192 run on the general kernel')
    run(kind, 4, 2, dim, vdim, SCHEDULES[schedule])


@pytest.mark.parametrize('kind', ['ruzinex', 'kept', 'tolenex'])
@pytest.mark.parametrize('steps', [[[('a', 260)]], [[('a', 390), ('b', 130)], [('b', 390), ('a', 65)]]], ids=['more', 'many'])
def test_many_workgroups(kind, steps):
    """64 heads: 260 rows make 320 workgroups of 64 rows, 390 beside 130 make 512 of 128."""
    run(kind, 64, 16, 64, 64, steps)


@pytest.mark.parametrize('steps', [[[('a', 260)]], [[('a', 390), ('b', 130)], [('b', 390), ('a', 65)]]], ids=['more', 'many'])
@pytest.mark.parametrize('kind,dim,vdim', [('ruzinex', 128, 128), ('kept', 128, 64), ('ruzinex', 192, 128), ('kept', 192, 64), ('window', 64, 128), ('tolenex', 128, 128)])
def test_many_workgroups_of_wider_heads(kind, dim, vdim, steps):
    """The same with heads of 128 and 192 query and 64 and 128 value dimensions."""
    run(kind, 64, 16, dim, vdim, steps)


@pytest.mark.parametrize('heads,steps', [(64, [[('a', 200)]]), (32, [[('a', 200), ('b', 90)]]), (32, [[('a', 700)]]), (32, [[('b', 130), ('a', 380)]])],
                         ids=['shared keys', 'shared keys, two', 'own keys', 'own keys, two'])
@pytest.mark.parametrize('kind,dim', [('tolenex', 64), ('ruzinex', 128)])
def test_levels_whose_order_turns(kind, dim, heads, steps):
    """Up to two workgroups on each of 256 CUs, the lightest first from the fifth (700 rows: the ninth) level of tiles on: two or three levels change places."""
    run(kind, heads, heads // 4, dim, dim, steps)


@pytest.mark.parametrize('page', [32, 128])
@pytest.mark.parametrize('kind', sorted(KINDS))
def test_pages_of_other_sizes(kind, page):
    run(kind, 4, 2, 64, 64, SCHEDULES['portions'], page)


@pytest.mark.parametrize('heads,steps', [(4, [[('a', 193)]]), (64, [[('a', 260)]]), (64, [[('b', 390), ('a', 130)]])], ids=['few', 'more', 'many'])
@pytest.mark.parametrize('where', [40, 100])
@pytest.mark.parametrize('kind', sorted(KINDS))
def test_a_row_without_finite_numbers_reaches_no_row_that_does_not_see_it(kind, heads, steps, where):
    """Row `where` of a request is NaN in every channel.  The rows before it, and with a window the ones that have left it behind, are what they
    are with another token in its place."""
    mod, cfg = KINDS[kind](heads, heads // 4 if heads == 64 else 2, 64, 64)
    toks, other = mod.tokens_for(cfg, sum(k for step in steps for rid, k in step if rid == 'a'), 3), mod.tokens_for(cfg, 390, 4)
    bad = next(t for t in range(cfg['vocab']) if t not in toks and t not in other)
    w = mod.random_weights(cfg, 13)
    finite = dict(w, embed=w['embed'].copy())
    w['embed'][bad] = np.nan
    toks[where] = bad
    reqs = {'a': toks, 'b': other}
    got = mod.replay(mod.session_for(cfg, w, 'bfloat16', max_tokens=2048), {r: reqs[r] for step in steps for r, _ in step}, steps)
    assert not np.isfinite(got['a'][where]).any()
    for rid, rows in got.items():
        sees = np.zeros(len(rows), bool)
        if rid == 'a':
            sees[where:where + 70 if kind == 'window' else None] = True
        if mod is test_gpu_vetipel:
            want = mod.O.logits(reqs[rid], as_f64(finite), cfg)
            mod.check(rows[~sees], want[~sees], mod.tol_of('bfloat16'), rid)
        else:
            n = int((~sees).sum())
            assert not sees[:n].any()
            if kind == 'ruzinex':  # (its head is its embedding: the bad token's own column is NaN in every row)
                rows[:n, bad] = mod.O.logits(reqs[rid][:n], as_f64(finite), cfg)[:, bad]
            mod.check_rows(rows[:n], reqs[rid][:n], finite, cfg, 'bfloat16', rid)
