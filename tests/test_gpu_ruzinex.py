"""Ruzinex through the ragged stack engine against the plain float64 oracle (oracle/ruzinex_oracle.py), on small configurations and
random weights made here.  fp32 engine: tight bound (what summation order can explain), routers with random weights (their decisions
are checked on the oracle not to be close calls at that bound); bfloat16 engine: loose bound, routers rigged so that no decision is
close, and crafted weights where random ones would hide a fault (one far key among hundreds and its mixed value, a sink, a lambda, the
shared expert's gate, a router's bias)."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest

from oracle import ruzinex_oracle as O
from ruzinex_cases import as_model, as_tensors, decisive_router, dense, layer, make_config, moe, random_weights, routed, routing_margin
from tolenex_cases import as_f64, bf16_round, rel_err, replay

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
F32_TOL, BF16_TOL = 3e-5, 5e-2


def weights_for(cfg, seed, dtype, toks=None):
    """Random weights; for the bfloat16 engine the routers are rigged.  With `toks`, the routers' decisions on them are checked on
    the oracle to stand clear of what the engine's rounding can move; a model with a close call is passed over for the next seed."""
    need = 0.1 if dtype == 'bfloat16' else 1e-4
    for attempt in range(20):
        w = random_weights(cfg, seed + 1000 * attempt)
        if not routed(cfg):
            return w
        if dtype == 'bfloat16':
            w = decisive_router(cfg, w, seed)
        if toks is None or all(routing_margin(cfg, w, t) > need for t in (toks.values() if isinstance(toks, dict) else [toks])):
            return w
    raise AssertionError('twenty models in a row with a router decision that is a close call')


def session_for(cfg, w, dtype='float32', max_tokens=1024, max_sequences=4, **kw):
    from tensorrt_llm.runtime import RaggedGenerationSession
    return RaggedGenerationSession(as_model(cfg, w), dtype=dtype, max_tokens=max_tokens, max_sequences=max_sequences, **kw)


def tokens_for(cfg, n, seed):
    return np.random.default_rng(seed).integers(0, cfg['vocab'], n).tolist()


def check(got, want, tol, what=''):
    e = rel_err(got, want)
    assert np.isfinite(got).all(), what
    assert e.max() < tol, f'{what}: worst row {int(e.argmax())} of {len(e)} has relative error {e.max():.3g} (bound {tol})'


def tol_of(dtype):
    return F32_TOL if dtype == 'float32' else BF16_TOL


def to_bf16(x):
    return bf16_round(np.asarray(x, np.float32)).astype(np.float64)


def check_rows(got, toks, w, cfg, dtype, what=''):
    """Every position of a request against the oracle.  fp32: the flat bound.  bfloat16: a row is held to 3 x the most that rounding the
    oracle's own activations to bfloat16 does to it, to nearest and with two random ditherings (never less than the median row's); no
    row may pass 1.5 x that, and at most one row in fifty (or one) may pass it at all."""
    wf = as_f64(w)
    want = O.logits(toks, wf, cfg)
    if dtype == 'float32':
        return check(got, want, F32_TOL, what)
    moved = np.zeros(len(toks))
    for seed in range(3):
        rng = np.random.default_rng(seed)
        fn = to_bf16 if seed == 0 else lambda x: to_bf16(x * (1.0 + rng.uniform(-2.0 ** -9, 2.0 ** -9, np.shape(x))))
        with O.rounding(fn):
            moved = np.maximum(moved, rel_err(O.logits(toks, wf, cfg), want))
    limit = 3.0 * np.maximum(moved, np.median(moved))
    e = rel_err(got, want)
    assert np.isfinite(got).all(), what
    worst = int((e / limit).argmax())
    assert (e < 1.5 * limit).all(), f'{what}: row {worst} of {len(e)} has relative error {e[worst]:.3g}, its limit is {limit[worst]:.3g}'
    assert (e > limit).sum() <= max(1, len(e) // 50), f'{what}: {(e > limit).sum()} of {len(e)} rows are over their limits'
    assert np.median(e) < 3e-2, f'{what}: the median row is off by {np.median(e):.3g}'


GENERAL = make_config([layer(v_mix=False, mlp=moe()), layer(heads=6, kv_heads=2, dim=10, vdim=24, rot_dims=10, mlp=dense()), layer(heads=3, kv_heads=3, dim=7, vdim=16, rot_dims=4, mlp=None),
                       layer(heads=2, kv_heads=1, dim=12, vdim=48, rot_dims=0, mlp=moe(experts=7, top=3, ff=10, shared=0)),
                       layer(mlp=moe(experts=3, top=1, ff=40, shared=9))], eps=3e-6)
# shapes the MFMA tile kernels and the LDS-staged products take in bfloat16; fp32 runs them on the general kernels
TILED = make_config([layer(heads=8, kv_heads=2, dim=64, vdim=32, rot_dims=32, mlp=moe(experts=8, top=3, ff=64, shared=128)),
                     layer(heads=6, kv_heads=2, dim=96, vdim=32, rot_dims=96, mlp=dense(ff=320)),
                     layer(heads=2, kv_heads=1, dim=32, vdim=64, rot_dims=16, mlp=moe(experts=4, top=2, ff=128, shared=64))], width=256, vocab=320)
STACKS = {'general': GENERAL, 'tiled': TILED}

MECHANISMS = {
    'attention_alone': make_config([layer()]),
    'attention_one_head': make_config([layer(heads=1, kv_heads=1, dim=8, vdim=5, rot_dims=8)]),
    'attention_one_kv_head': make_config([layer(heads=5, kv_heads=1, dim=6, vdim=10, rot_dims=2)]),
    'attention_kv_per_head': make_config([layer(heads=3, kv_heads=3)]),
    'attention_values_wider_than_keys': make_config([layer(heads=4, dim=4, vdim=40, rot_dims=4)]),
    'attention_keys_wider_than_values': make_config([layer(heads=4, dim=40, vdim=4, rot_dims=20)]),
    'attention_odd_key_size': make_config([layer(dim=9, vdim=7, rot_dims=6)], width=72),
    'attention_no_rotation': make_config([layer(rot_dims=0)]),
    'attention_fully_rotated': make_config([layer(rot_dims=16)]),
    'attention_one_pair_turns': make_config([layer(rot_dims=2)]),
    'attention_no_frequency_scaling': make_config([layer(factor=None)]),
    'attention_large_frequency_scaling': make_config([layer(factor=8.0, base=10.0)]),
    'attention_large_scale': make_config([layer(scale=1.0)]),
    'attention_wide_keys': make_config([layer(heads=2, kv_heads=1, dim=300, vdim=16, rot_dims=128)]),
    'mixing_everywhere': make_config([layer(), layer(), layer()]),
    'mixing_nowhere': make_config([layer(v_mix=False), layer(v_mix=False)]),
    'mixing_in_one_layer': make_config([layer(v_mix=False), layer(), layer(v_mix=False)]),
    'mixing_from_the_second_layer_on': make_config([layer(v_mix=False), layer(), layer(v_mix=False), layer()]),
    'mixing_across_head_shapes': make_config([layer(heads=4, kv_heads=4, vdim=12), layer(heads=2, kv_heads=2, vdim=24), layer(heads=3, kv_heads=1, vdim=48)]),
    'dense_alone': make_config([layer(heads=1, kv_heads=1, dim=4, vdim=4, rot_dims=4, mlp=dense())]),
    'dense_odd_size': make_config([layer(mlp=dense(ff=37))]),
    'dense_unaligned_rows': make_config([layer(mlp=dense(ff=100))], width=128),
    'dense_tile_sizes': make_config([layer(mlp=dense(ff=256))], width=128),
    'moe_alone': make_config([layer(heads=1, kv_heads=1, dim=4, vdim=4, rot_dims=4, mlp=moe())]),
    'moe_no_shared': make_config([layer(mlp=moe(shared=0))]),
    'moe_top_one': make_config([layer(mlp=moe(experts=5, top=1))]),
    'moe_one_expert': make_config([layer(mlp=moe(experts=1, top=1))]),
    'moe_every_expert': make_config([layer(mlp=moe(experts=4, top=4))]),
    'moe_many_experts': make_config([layer(mlp=moe(experts=70, top=5, ff=9, shared=8))], width=160),
    'moe_sixteen_chosen': make_config([layer(mlp=moe(experts=20, top=16, ff=8, shared=16))], width=128),
    'moe_equal_shared_and_expert_size': make_config([layer(mlp=moe(ff=32, shared=32))]),
    'moe_odd_sizes': make_config([layer(mlp=moe(experts=5, top=2, ff=13, shared=21))]),
    'moe_tile_sizes': make_config([layer(heads=2, dim=32, vdim=32, mlp=moe(experts=4, top=2, ff=128, shared=192))], width=128),
    'moe_tile_sizes_no_shared': make_config([layer(heads=2, dim=32, vdim=32, mlp=moe(experts=4, top=2, ff=192, shared=0))], width=128),
    'moe_shared_ends_inside_a_tile': make_config([layer(heads=2, dim=32, vdim=32, mlp=moe(experts=4, top=2, ff=64, shared=72))], width=128),
    'moe_shared_rows_unaligned': make_config([layer(heads=2, dim=32, vdim=32, mlp=moe(experts=4, top=2, ff=52, shared=44))], width=128),
    'residual_unscaled': make_config([layer(mlp=dense()), layer(mlp=moe())], mult=1.0),
    'residual_amplified': make_config([layer(mlp=dense()), layer()], mult=1.8),
    'no_feed_forward_in_the_last_layer': make_config([layer(mlp=moe()), layer(mlp=None)]),
    'large_eps': make_config([layer(mlp=moe())], eps=0.3),
    'width_that_is_no_multiple_of_four': make_config([layer(heads=3, kv_heads=1, dim=7, vdim=5, rot_dims=6, mlp=moe(experts=5, top=2, ff=10, shared=7)),
                                                      layer(heads=2, kv_heads=1, dim=9, vdim=5, rot_dims=2, mlp=dense(ff=11))], width=70, vocab=131),
    'general_stack': GENERAL,
    'tiled_stack': TILED,
}
for _d in (32, 64, 96, 128, 192):
    for _v in (32, 64, 96, 128):
        MECHANISMS[f'attention_tile_{_d}_{_v}'] = make_config([layer(heads=6, kv_heads=2 if _v != 64 else 1, dim=_d, vdim=_v, rot_dims=_d // 2)], width=128)


@pytest.mark.parametrize('name', sorted(MECHANISMS))
@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
def test_each_mechanism_whole_prompt(name, dtype):
    cfg = MECHANISMS[name]
    toks = tokens_for(cfg, 150, 1)  # crosses page borders
    w = weights_for(cfg, len(name), dtype, toks)
    s = session_for(cfg, w, dtype)
    got = replay(s, {'a': toks}, [[('a', len(toks))]])['a']
    check_rows(got, toks, w, cfg, dtype, name)


@pytest.mark.parametrize('name', sorted(MECHANISMS))
@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
def test_each_mechanism_decoded(name, dtype):
    cfg = MECHANISMS[name]
    toks = tokens_for(cfg, 75, 2)
    w = weights_for(cfg, len(name) + 1, dtype, toks)
    s = session_for(cfg, w, dtype)
    got = replay(s, {'a': toks}, [[('a', 60)], [('a', 2)]] + [[('a', 1)]] * 13)['a']
    check_rows(got, toks, w, cfg, dtype, name)


@pytest.mark.parametrize('stack', sorted(STACKS))
@pytest.mark.parametrize('dtype,bound', [('float32', 1e-5), ('bfloat16', 5e-2)])
def test_residual_stream_behind_every_layer(stack, dtype, bound):
    cfg = STACKS[stack]
    toks = tokens_for(cfg, 19, 2)
    w = weights_for(cfg, 3, dtype, toks)
    _, taps = O.forward(toks, as_f64(w), cfg, return_layers=True)
    s = session_for(cfg, w, dtype, debug_mode=True)
    s.step([('a', toks, [0])])
    assert s.engine.layer_runs == len(taps) == len(cfg['layers'])
    for j, x in enumerate(taps):
        assert np.abs(s.engine.tap(j) - x).max() < bound * np.abs(x).max(), f'layer {j}'


@pytest.mark.parametrize('stack', sorted(STACKS))
@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
def test_prefill_then_token_by_token(dtype, stack):
    cfg = STACKS[stack]
    toks = tokens_for(cfg, 170, 3)
    w = weights_for(cfg, 5, dtype, toks)
    s = session_for(cfg, w, dtype)
    got = replay(s, {'a': toks}, [[('a', 100)]] + [[('a', 1)]] * 70)['a']
    check_rows(got, toks, w, cfg, dtype)


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('sizes', [[2] * 40, [3, 61, 2, 64, 1, 5, 2, 58, 1, 1, 2], [63, 2, 63, 1, 1, 66], [1] * 9 + [120, 2], [8, 9, 31, 32, 33, 7, 40]])
@pytest.mark.parametrize('stack', sorted(STACKS))
def test_portions_of_a_prompt(sizes, dtype, stack):
    cfg = STACKS[stack]
    toks = tokens_for(cfg, sum(sizes), 4)
    w = weights_for(cfg, 8, dtype, toks)
    s = session_for(cfg, w, dtype)
    got = replay(s, {'a': toks}, [[('a', n)] for n in sizes])['a']
    check_rows(got, toks, w, cfg, dtype)


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('stack', sorted(STACKS))
def test_unequal_requests_in_one_batch_equal_each_alone(dtype, stack):
    cfg = STACKS[stack]
    reqs = {'a': tokens_for(cfg, 131, 5), 'b': tokens_for(cfg, 9, 6), 'c': tokens_for(cfg, 66, 7), 'd': tokens_for(cfg, 2, 8)}
    w = weights_for(cfg, 9, dtype, reqs)
    schedule = [[('a', 60), ('b', 2)], [('b', 1), ('a', 5), ('c', 64)], [('c', 1), ('b', 1), ('a', 1), ('d', 2)],
                [('a', 63), ('b', 5), ('c', 1)], [('a', 1)], [('a', 1)]]
    s = session_for(cfg, w, dtype)
    got = replay(s, reqs, schedule)
    for rid, toks in reqs.items():
        check_rows(got[rid], toks, w, cfg, dtype, rid)
        alone = replay(s, {rid: toks}, [[(rid, len(toks))]])[rid]
        check(got[rid], alone, 2e-5 if dtype == 'float32' else BF16_TOL, f'{rid} alone')
    assert not s.live() and s.cache.blocks_manager.num_free_blocks() == s.num_blocks and s.slots.num_free_slots() == 4


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
def test_requests_of_very_unequal_length_decode_side_by_side(dtype):
    """Contexts from 1 to 700 tokens in one decoding step: the key split over workgroups leaves empty shares to the short ones."""
    cfg = TILED
    reqs = {'long': tokens_for(cfg, 718, 90), 'mid': tokens_for(cfg, 75, 91), 'new': tokens_for(cfg, 12, 92)}
    w = weights_for(cfg, 21, dtype, reqs)
    schedule = [[('long', 698)], [('mid', 65), ('long', 1)]] + [[('long', 1), ('mid', 1), ('new', 1)]] * 10 + [[('long', 9), ('new', 2)]]
    s = session_for(cfg, w, dtype, max_tokens=1024)
    got = replay(s, reqs, schedule)
    for rid, toks in reqs.items():
        check_rows(got[rid], toks, w, cfg, dtype, rid)


@pytest.mark.parametrize('wide', ['0', '1'])
def test_both_prompt_forms_of_wide_keys(wide, monkeypatch):
    monkeypatch.setenv('TLLM_STACK_WIDE_PREFILL', wide)
    cfg = make_config([layer(heads=6, kv_heads=2, dim=192, vdim=128, rot_dims=96), layer(heads=4, kv_heads=2, dim=192, vdim=128, rot_dims=192, mlp=moe())], width=128)
    reqs = {'a': tokens_for(cfg, 300, 95), 'b': tokens_for(cfg, 171, 96)}
    w = weights_for(cfg, 25, 'bfloat16', reqs)
    schedule = [[('a', 129), ('b', 33)], [('a', 1), ('b', 130)], [('a', 150), ('b', 1)], [('a', 20), ('b', 7)]]
    s = session_for(cfg, w, 'bfloat16')
    got = replay(s, reqs, schedule)
    for rid, toks in reqs.items():
        check_rows(got[rid], toks, w, cfg, 'bfloat16', rid)


@pytest.mark.parametrize('mlp', [dense(ff=3000), dense(ff=6000), dense(ff=8000), moe(experts=2, top=2, ff=1536, shared=3000), moe(experts=3, top=3, ff=1544, shared=1003),
                                 moe(experts=2, top=2, ff=64, shared=6000)], ids=lambda m: f"{m['kind']}{m.get('ff') or (m['expert']['ff'], m['shared']['ff'])}")
def test_gated_products_of_every_tile_shape(mlp):
    """Feed-forwards wide enough, over prompts long enough, that the products take several of the tile shapes (every one, over more lengths of K:
    test_gpu_product_tiles.py); the columns behind the shared expert's start inside a tile."""
    cfg = make_config([layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=mlp)], width=64)
    toks = tokens_for(cfg, 1000, 97)
    w = random_weights(cfg, 98)
    check_rows(replay(session_for(cfg, w, 'bfloat16'), {'a': toks}, [[('a', 1000)]])['a'], toks, w, cfg, 'bfloat16')


def test_pages_and_slots_that_are_used_again():
    """A pool of 4 pages and 2 slots serves six requests one after another and side by side: every page is written by several
    requests, and what an earlier one left there must never be seen by a later one."""
    cfg = GENERAL
    every = {f'{n}{r}': tokens_for(cfg, *a) for r in range(3) for n, a in (('x', (100 + r, 20 + r)), ('y', (70 - r, 30 + r)))}
    w = weights_for(cfg, 11, 'float32', every)
    s = session_for(cfg, w, 'float32', max_tokens=256, max_sequences=2)
    assert s.num_blocks == 4
    used_blocks, used_slots = [], []
    for rnd in range(3):
        x, y = f'x{rnd}', f'y{rnd}'
        reqs = {k: every[k] for k in (x, y)}
        schedule = [[(x, 50), (y, 3)], [(y, len(reqs[y]) - 3), (x, 1)], [(x, len(reqs[x]) - 51)]]
        got = replay(s, reqs, schedule, end_when_done=False)
        for rid in reqs:
            seq = s._seq[rid]
            used_blocks.append(tuple(s.cache.blocks_manager.block_ids(seq)[0]))
            used_slots.append(s.slots.slot_of(seq))
            check(got[rid], O.logits(reqs[rid], as_f64(w), cfg), F32_TOL, rid)
            s.release(rid)
    assert len(set(used_slots)) == 2 and len(used_slots) == 6
    assert len({b for blocks in used_blocks for b in blocks}) == 4 and sum(len(b) for b in used_blocks) == 12


# ------------------------------------------------------------------------------------------------ rigged weights
def rigged(n, p_far, seed, heads=4, kv_heads=2, D=16, E=24, rot_dims=8):
    """Two mixing layers; head 0 of the second is rigged so that the LAST token's query meets the key of the token at p_far with a score
    far above all others, so that dropping, shifting or corrupting it - or the first layer's value of that token, of which the cached
    value is mostly made - moves the logits at the last position by much more than bfloat16 rounding: channels 0 and 1 of the residual
    belong to the far and to the last token (no sublayer lands there), and the last dimension of head 0's query and key, which does not
    turn, reads nothing else."""
    cfg = make_config([layer(heads=heads, kv_heads=kv_heads, dim=D, vdim=E, rot_dims=rot_dims), layer(heads=heads, kv_heads=kv_heads, dim=D, vdim=E, rot_dims=rot_dims)])
    w = random_weights(cfg, seed)
    rng = np.random.default_rng(seed)
    far_tok = 3
    last_tok = far_tok if p_far == n - 1 else 4
    toks = [int(t) for t in rng.integers(5, cfg['vocab'], n)]
    toks[p_far], toks[-1] = far_tok, last_tok
    w['embed'][:, :2] = 0.0
    w['embed'][far_tok, 0] = w['embed'][last_tok, 1] = 20.0
    w['l0.mix.vmix'] = bf16_round(np.float32(0.0))
    w['l1.mix.vmix'] = bf16_round(np.float32(0.75))
    w['l0.norm1b'][:2] = 0.0
    w['l1.norm1'][:2] = 1.0
    for name, ch, g in (('k', 0, 4.0), ('q', 1, 0.8 / cfg['layers'][1]['mixer']['scale'])):
        w['l1.mix.' + name][D - 1] = 0.0
        w['l1.mix.' + name][D - 1, ch] = bf16_round(np.float32(g))
        w[f'l1.mix.{name}.b'][D - 1] = 0.0
    w['l1.mix.sink'][0] = 2.0
    w['l1.norm1b'] *= 2.0
    return cfg, w, toks


@pytest.mark.parametrize('p_far', [0, 1, 31, 32, 63, 64, 127, 128, 200, 331])
@pytest.mark.parametrize('dtype,shape', [('float32', (4, 2, 16, 24, 8)), ('bfloat16', (4, 2, 16, 24, 8)), ('bfloat16', (8, 1, 64, 32, 32)), ('bfloat16', (6, 2, 96, 64, 48))])
def test_a_far_key_that_decides_the_answer(p_far, dtype, shape):
    """In a whole prompt, in a portion that starts behind the far token, decoded alone, and decoded beside another request."""
    cfg, w, toks = rigged(333, p_far, 40 + p_far, *shape)
    n, wf = len(toks), as_f64(w)
    want = O.logits(toks, wf, cfg)
    other = list(toks)
    other[p_far] = 7
    assert rel_err(O.logits(other, wf, cfg)[-1:], want[-1:])[0] > 0.1, 'the rig does not bite: the far token does not decide'
    for wrong in (0.0, 1.0):
        moved = rel_err(O.logits(toks, dict(wf, **{'l1.mix.vmix': np.float64(wrong)}), cfg)[-1:], want[-1:])[0]
        assert moved > 0.1 * abs(wrong - 0.75), f'the rig does not bite: lambda {wrong} moves the last row by {moved:.3g} only'
    s = session_for(cfg, w, dtype)
    cut = max(p_far + 1, 2)
    check(replay(s, {'w': toks}, [[('w', n)]])['w'][-1:], want[-1:], tol_of(dtype), 'whole')
    check(replay(s, {'p': toks}, [[('p', cut)], [('p', n - cut)]])['p'][-1:], want[-1:], tol_of(dtype), 'portion')
    check(replay(s, {'d': toks}, [[('d', n - 1)], [('d', 1)]])['d'][-1:], want[-1:], tol_of(dtype), 'decoded')
    side = tokens_for(cfg, 4, 77)
    got = replay(s, {'d': toks, 'e': side}, [[('e', 3), ('d', 50)], [('d', n - 51)], [('e', 1), ('d', 1)]])
    check(got['d'][-1:], want[-1:], tol_of(dtype), 'decoded in a batch')


def moved_by(cfg, w, toks, **change):
    wf = as_f64(w)
    return np.median(rel_err(O.logits(toks, dict(wf, **{k.replace('__', '.'): np.asarray(v, np.float64) for k, v in change.items()}), cfg), O.logits(toks, wf, cfg)))


@pytest.mark.parametrize('heads,kv_heads,dim,vdim', [(6, 2, 16, 24), (12, 1, 64, 32), (24, 3, 32, 32), (40, 1, 32, 64)])
@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
def test_the_sinks_take_their_shares(dtype, heads, kv_heads, dim, vdim):
    """Sinks as large as the scores and different per head: leaving them out, or handing a head its neighbour's, changes the oracle's
    logits by much; whole prompt, then decoding (where the heads of a group are the rows of a tile)."""
    cfg = make_config([layer(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim)], mult=1.0)
    w = random_weights(cfg, 33)
    w['l0.mix.sink'][:] = bf16_round(np.linspace(1.0, 8.0, heads).astype(np.float32))
    w['l0.norm1b'] *= 2.0
    toks = tokens_for(cfg, 70, 34)
    for wrong in (np.full(heads, -1e9), np.roll(w['l0.mix.sink'], heads // 2)):
        assert moved_by(cfg, w, toks, l0__mix__sink=wrong) > 0.1
    s = session_for(cfg, w, dtype)
    check_rows(replay(s, {'a': toks}, [[('a', 40)]] + [[('a', 1)]] * 30)['a'], toks, w, cfg, dtype)


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
def test_what_belongs_to_one_layer_stays_there(dtype):
    """Lambdas, router biases and the shared expert's gate, large and different per layer: exchanging them, or leaving one out, moves the
    oracle's logits by much."""
    cfg = make_config([layer(mlp=moe(experts=4, top=4)), layer(mlp=moe(experts=4, top=4)), layer(mlp=moe(experts=4, top=4))], mult=1.0)
    w = random_weights(cfg, 37)
    for i, lam in enumerate((0.9, -0.6, 1.4)):
        w[f'l{i}.mix.vmix'] = bf16_round(np.float32(lam))
        w[f'l{i}.mlp.router.b'] = bf16_round(np.roll(np.array([3.0, 0.0, -2.0, 1.0], np.float32), i))
        w[f'l{i}.mlp.shared.sg'] = w[f'l{i}.mlp.shared.sg'] * 4.0
    toks = tokens_for(cfg, 40, 38)
    assert moved_by(cfg, w, toks, l1__mix__vmix=1.4, l2__mix__vmix=-0.6) > 0.1
    assert moved_by(cfg, w, toks, l1__mlp__router__b=w['l2.mlp.router.b'], l2__mlp__router__b=w['l1.mlp.router.b']) > 0.1
    assert moved_by(cfg, w, toks, l0__mlp__router__b=np.zeros(4)) > 0.05
    assert moved_by(cfg, w, toks, l0__mlp__shared__sg=-w['l0.mlp.shared.sg']) > 0.1
    s = session_for(cfg, w, dtype)
    check_rows(replay(s, {'a': toks}, [[('a', 30)]] + [[('a', 1)]] * 10)['a'], toks, w, cfg, dtype)


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('dim,vdim,rot', [(16, 24, 16), (64, 32, 64), (96, 64, 32)])
def test_pairs_frequencies_and_biases_of_the_rotation(dtype, dim, vdim, rot):
    """Large biases of q and k make the scores depend on the turn between them alone: other pairs, an undivided frequency, or a bias
    added behind the rotation would move every row."""
    cfg = make_config([layer(dim=dim, vdim=vdim, rot_dims=rot, base=100.0, factor=2.0, scale=0.5 / dim ** 0.5)], mult=1.0)
    w = random_weights(cfg, 39)
    for n in 'qk':
        w[f'l0.mix.{n}.b'] = w[f'l0.mix.{n}.b'] * 4.0
        w[f'l0.mix.{n}'] = w[f'l0.mix.{n}'] * 0.5
    toks = tokens_for(cfg, 130, 40)
    other = json.loads(json.dumps(cfg))
    other['layers'][0]['mixer']['rot']['scaling']['factor'] = 1.0
    wf = as_f64(w)
    assert np.median(rel_err(O.logits(toks, wf, other), O.logits(toks, wf, cfg))) > 0.05
    s = session_for(cfg, w, dtype)
    check_rows(replay(s, {'a': toks}, [[('a', 80)]] + [[('a', 1)]] * 50)['a'], toks, w, cfg, dtype)


@pytest.mark.parametrize('stack', sorted(STACKS))
def test_first_tokens_of_a_sequence(stack):
    cfg = STACKS[stack]
    lists = {n: tokens_for(cfg, n, 50 + n) for n in (1, 2, 3, 4, 5)}
    for dtype in ('float32', 'bfloat16'):
        w = weights_for(cfg, 13, dtype, lists)
        s = session_for(cfg, w, dtype)
        for n, toks in lists.items():
            want = O.logits(toks, as_f64(w), cfg)
            check(replay(s, {n: toks}, [[(n, n)]])[n], want, tol_of(dtype), f'{n} tokens at once')
            check(replay(s, {-n: toks}, [[(-n, 1)]] * n)[-n], want, tol_of(dtype), f'{n} tokens one by one')


@pytest.mark.parametrize('stack', sorted(STACKS))
def test_long_decoding(stack):
    cfg = STACKS[stack]
    toks = tokens_for(cfg, 330, 9)
    for dtype in ('float32', 'bfloat16'):
        w = weights_for(cfg, 15, dtype, toks)
        s = session_for(cfg, w, dtype)
        check_rows(replay(s, {'a': toks}, [[('a', 2)]] + [[('a', 1)]] * 328)['a'], toks, w, cfg, dtype, dtype)


# ------------------------------------------------------------------------------------------------ the options beside other ones
class DescribedModel(object):
    """An engine configuration and weights, served by a session like a model of the registry."""
    page_size = 64

    def __init__(self, config, w):
        self.config, self.w = config, w

    def build_stack_engine(self, dtype, num_blocks, num_slots, debug_taps=False, build_if_missing=False):
        from tensorrt_llm.runtime.stack import StackEngine
        return StackEngine(dict(self.config, dtype=dtype, num_blocks=num_blocks, num_slots=num_slots, debug_taps=int(debug_taps)), as_tensors(self.w))


def run_described(ec, w, dtype, toks):
    from tensorrt_llm.runtime import RaggedGenerationSession
    s = RaggedGenerationSession(DescribedModel(ec, w), dtype=dtype, max_tokens=256)
    return replay(s, {'a': toks}, [[('a', len(toks) - 10)]] + [[('a', 1)]] * 10)['a']


def described(cfg, **change):
    c = as_model(cfg, {}).config.engine_config()
    c.update({k.replace('__', '.'): v for k, v in change.items()})
    return c


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
def test_sublayers_that_land_without_a_norm(dtype):
    """post_norm=0: x <- x + m mixer(n1 x), x <- x + m ff(n2 x)."""
    cfg = make_config([layer(mlp=dense()), layer(mlp=moe(experts=3, top=3))], mult=0.4)
    w = random_weights(cfg, 61)
    toks = tokens_for(cfg, 80, 62)
    wf, x, first = as_f64(w), as_f64(w)['embed'][toks], None
    for i, l in enumerate(cfg['layers']):
        y, first = O.attention(O.rms_norm(x, wf[f'l{i}.norm1'], 1e-5), wf, f'l{i}.mix.', l['mixer'], first)
        x = x + 0.4 * y
        x = x + 0.4 * O.feed_forward(O.rms_norm(x, wf[f'l{i}.norm2'], 1e-5), wf, f'l{i}.mlp.', l['mlp'])
    want = O.rms_norm(x, wf['final.norm'], 1e-5) @ wf['embed'].T
    check(run_described(described(cfg, post_norm=0), {k: v for k, v in w.items() if not k.endswith(('1b', '2b'))}, dtype, toks), want, tol_of(dtype))


@pytest.mark.parametrize('experts', ['silu_gate', 'relu2'])
@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
def test_gated_shared_experts_behind_a_hyper_connected_residual(dtype, experts):
    """Two copies of the stream that start alike, connected by identities: the plain pre-norm sum; both forms of the experts."""
    cfg = make_config([layer(mlp=moe(experts=3, top=3))])
    w = random_weights(cfg, 63)
    if experts == 'relu2':
        w = {k: v for k, v in w.items() if '.mlp.' not in k or not k.endswith('.gate')}
    for q in ('hc1', 'hc2'):
        w[f'l0.{q}.in'], w[f'l0.{q}.out'], w[f'l0.{q}.mix'] = np.array([0.5, 0.5], np.float32), np.array([1.0, 1.0], np.float32), np.eye(2, dtype=np.float32)
    toks = tokens_for(cfg, 80, 64)
    wf = as_f64(w)
    x = wf['embed'][toks]
    x = x + O.attention(O.rms_norm(x, wf['l0.norm1'], 1e-5), wf, 'l0.mix.', cfg['layers'][0]['mixer'], None)[0]
    h, p = O.rms_norm(x, wf['l0.norm2'], 1e-5), 'l0.mlp.'

    def expert(n):
        if experts == 'silu_gate':
            return O.gated_ff(h, wf, p + n, O.silu)
        return np.maximum(h @ wf[p + n + 'up'].T, 0.0) ** 2 @ wf[p + n + 'down'].T

    chosen, g = O.route(h, wf, p, {'top': 3})
    ff = O.sigmoid(h @ wf[p + 'shared.sg'].T) * expert('shared.')
    for e in range(3):
        ff = ff + np.where(chosen == e, g, 0.0).sum(axis=1, keepdims=True) * expert(f'e{e}.')
    want = 2.0 * (x + ff)  # the output norm reads the sum of the copies
    want = O.rms_norm(want, wf['final.norm'], 1e-5) @ wf['embed'].T
    ec = described(cfg, residual='hyper', streams=2, post_norm=0, residual_mult=1, loop_input=1, layer__0__expert=experts)
    check(run_described(ec, w, dtype, toks), want, tol_of(dtype))


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('dim,rot', [(16, 10), (130, 130), (64, 64)])
def test_half_split_pairs_behind_a_norm_of_q_and_k(dtype, dim, rot):
    """Weighted unit-RMS queries and keys, then half-split pairs (a wave per head), value mixing beside them."""
    cfg = make_config([layer(dim=dim, rot_dims=rot), layer(dim=dim, rot_dims=rot)])
    w = random_weights(cfg, 65)
    rng = np.random.default_rng(66)
    for i in range(2):
        for n in 'qk':
            w[f'l{i}.mix.{n}.norm'] = bf16_round(rng.standard_normal(dim).astype(np.float32) * 0.2 + 1.0)
    toks = tokens_for(cfg, 80, 67)
    wf = as_f64(w)
    x, first = wf['embed'][toks], None
    for i, l in enumerate(cfg['layers']):
        p, m = f'l{i}.mix.', l['mixer']
        h = O.rms_norm(x, wf[f'l{i}.norm1'], 1e-5)
        q, k, v = [(h @ wf[p + c].T + wf[p + c + '.b']).reshape(len(toks), -1, n) for c, n in (('q', dim), ('k', dim), ('v', m['vdim']))]
        q, k = [O.rotate_half(O.rms_norm(a, wf[p + n + '.norm'], 1e-5), m['rot']) for a, n in ((q, 'q'), (k, 'k'))]
        v, first = (v, v) if first is None else (O.mix_values(v, first, float(wf[p + 'vmix'])), first)
        ctx = [O.sink_softmax(q[:, a] @ k[:, a // 2].T * m['scale'], float(wf[p + 'sink'][a])) @ v[:, a // 2] for a in range(4)]
        x = x + 0.6 * O.rms_norm(np.concatenate(ctx, axis=1) @ wf[p + 'o'].T, wf[f'l{i}.norm1b'], 1e-5)
    want = O.rms_norm(x, wf['final.norm'], 1e-5) @ wf['embed'].T
    ec = described(cfg, **{f'layer__{i}__{k}': 1 for i in range(2) for k in ('qk_norm', 'qk_norm_weight')})
    check(run_described(ec, w, dtype, toks), want, tol_of(dtype))


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
def test_a_window_a_normed_embedding_and_a_loop(dtype):
    """What the sandwich-normed block takes from its neighbours: a window mask, a normed embedding row, a range of layers that runs twice
    (a cache per pass, its step ahead of the first layer), a head of its own."""
    cfg = make_config([layer(v_mix=False, mlp=dense()), layer(v_mix=False, mlp=moe(experts=2, top=2))])
    w = random_weights(cfg, 68)
    rng = np.random.default_rng(69)
    W = cfg['width']
    w['embed.norm'] = bf16_round(rng.standard_normal(W).astype(np.float32) * 0.2 + 1.0)
    w['loop.step'] = bf16_round(rng.standard_normal((2, W)).astype(np.float32))
    w['head'] = bf16_round(rng.standard_normal((cfg['vocab'], W)).astype(np.float32))
    toks = tokens_for(cfg, 90, 70)
    wf = as_f64(w)
    x = O.rms_norm(wf['embed'][toks], wf['embed.norm'], 1e-5)
    near = np.subtract.outer(np.arange(90), np.arange(90)) < 20
    plain = O.sink_softmax
    try:
        O.sink_softmax = lambda s, sink: plain(np.where(near, s, -1e30), sink)
        for t in range(2):
            x = x + wf['loop.step'][t]
            for i in range(2):
                x, _ = O.layer_forward(x, wf, cfg, i, None)
    finally:
        O.sink_softmax = plain
    want = O.rms_norm(x, wf['final.norm'], 1e-5) @ wf['head'].T
    ec = described(cfg, embedding_norm=1, tied_head=0, loop_start=0, loop_stop=2, loop_times=2,
                   **{f'layer__{i}__{k}': v for i in range(2) for k, v in (('mask', 'window'), ('mask_size', 20))})
    check(run_described(ec, w, dtype, toks), want, tol_of(dtype))


def test_descriptions_that_cannot_run_are_refused():
    from tensorrt_llm.runtime.stack import StackEngine
    cfg = make_config([layer(mlp=moe()), layer(mlp=dense())])
    w = random_weights(cfg, 45)
    good = described(cfg, dtype='float32', num_blocks=2, num_slots=1)
    for change in ({'block': 'parallel'}, {'residual': 'gated'}, {'residual': 'hyper', 'loop_input': 1}, {'norm_groups': 3}, {'loop_input': 1}, {'layer.0.rot_pairing': 'other'},
                   {'layer.0.rot_dims': 7}, {'layer.1.vdim': 25}, {'loop_stop': 2, 'loop_times': 2}, {'layer.0.shared_ff': 0}, {'token_side': 4},
                   {'layer.0.rot_scaling': 'cubic'}, {'layer.0.kv_heads': 3}):
        with pytest.raises(RuntimeError):
            StackEngine(dict(good, **change), as_tensors(w))
    for name in ('l1.norm2b', 'l0.mlp.shared.sg', 'l1.mix.vmix', 'l0.mlp.router.b', 'l0.mix.k.b'):
        with pytest.raises(RuntimeError, match=name.replace('.', r'\.')):
            StackEngine(good, as_tensors({k: v for k, v in w.items() if k != name}))


SMALL = make_config([layer(heads=2, mlp=moe(experts=4, top=2, ff=16, shared=24)), layer(heads=4, mlp=dense(ff=40)), layer(heads=2, mlp=moe(experts=3, top=1, ff=20, shared=0))],
                    width=64, vocab=97)


def test_greedy_generation_through_the_scheduler():
    """Six prompts, four slots, 40 tokens per step: prompts are cut, requests queue, decoded tokens share steps with prompt portions.
    fp32 engine against the oracle's greedy continuation (recomputed from scratch for every token)."""
    from tensorrt_llm.runtime import SamplingConfig
    cfg = SMALL
    w = random_weights(cfg, seed=17)
    prompts = [tokens_for(cfg, n, 60 + n) for n in (70, 3, 45, 1, 90, 17)]
    s = session_for(cfg, w, 'float32', max_tokens=512, max_sequences=4, max_batch_tokens=40)
    outs = s.decode_batch(prompts, SamplingConfig(end_id=-1, pad_id=0), max_new_tokens=6)
    for p, o in zip(prompts, outs):
        assert o.tolist() == O.greedy(p, as_f64(w), cfg, 6)
    assert not s.live() and s.cache.blocks_manager.num_free_blocks() == s.num_blocks


def test_command_lines(tmp_path):
    """examples/ruzinex/run.py generates from a checkpoint directory; bin/trace_run replays a recorded schedule from it."""
    from test_gpu_tolenex import write_checkpoint
    cfg = SMALL
    w = random_weights(cfg, seed=19)
    ck = str(tmp_path / 'ck')
    write_checkpoint(ck, cfg, w)
    prompt = tokens_for(cfg, 21, 70)
    np.save(tmp_path / 'in.npy', np.asarray(prompt, np.int32))
    run = os.path.join(ROOT, 'trtllm-llama_amd', 'examples', 'ruzinex', 'run.py')
    subprocess.run([sys.executable, run, '--model_dir', ck, '--dtype', 'float32', '--input_tokens', str(tmp_path / 'in.npy'),
                    '--max_output_len', '5', '--output_npy', str(tmp_path / 'out.npy')], check=True, timeout=300)
    assert np.load(tmp_path / 'out.npy').reshape(-1)[len(prompt):].tolist() == O.greedy(prompt, as_f64(w), cfg, 5)
    a, b = tokens_for(cfg, 70, 71), tokens_for(cfg, 5, 72)
    steps = [{'step': 0, 'entries': [{'id': 'a', 'tokens': a[:66], 'want': [0, 65]}, {'id': 'b', 'tokens': b[:2], 'want': []}], 'end': []},
             {'step': 1, 'entries': [{'id': 'b', 'tokens': b[2:], 'want': [2]}], 'end': ['b']},
             {'step': 2, 'entries': [{'id': 'a', 'tokens': a[66:], 'want': [3]}], 'end': ['a']}]
    out = tmp_path / 'logits'
    r = subprocess.run([os.path.join(ROOT, 'bin', 'trace_run'), '--model', ck, '--dtype', 'float32', '--out', str(out), '--max-tokens', '192'],
                       input='\n'.join(json.dumps(s) for s in steps) + '\n', capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    assert [l for l in r.stdout.splitlines() if l.startswith('done')] == ['done 0', 'done 1', 'done 2']
    la, lb = O.logits(a, as_f64(w), cfg), O.logits(b, as_f64(w), cfg)
    check(np.fromfile(out / '0.f32', '<f4').reshape(2, -1), la[[0, 65]], F32_TOL)
    check(np.fromfile(out / '1.f32', '<f4').reshape(1, -1), lb[[4]], F32_TOL)
    check(np.fromfile(out / '2.f32', '<f4').reshape(1, -1), la[[69]], F32_TOL)
