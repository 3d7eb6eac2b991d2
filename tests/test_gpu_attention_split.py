"""Attention of decoded tokens (attn_tile_kernel of stack_attn.hip) around the context at which its keys are split over workgroups, one block of 32 keys
to a wave of the first: contexts of 26 .. 38, 122 .. 134 and 250 .. 262 keys, two maps a head with and without a soft cap, windows with kept keys, and
two requests beside each other of which the short one leaves splits empty.  Bounds as in the designs' own tests."""
import pytest

import narurax_cases as NC
import test_gpu_narurax as N
import test_gpu_tolenex as GT
import tolenex_cases as T

pytestmark = pytest.mark.gpu

STARTS = [26, 122, 250]
STEPS = [[('a', 1)]] * 5 + [[('a', 1), ('b', 1)]] * 7


def requests(G, cfg, start):
    reqs = {'a': G.tokens_for(cfg, start + 12, 31), 'b': G.tokens_for(cfg, 10, 32)}
    return reqs, [[('a', start)], [('b', 3)]] + STEPS


@pytest.mark.parametrize('start', STARTS)
@pytest.mark.parametrize('softcap', [30.0, 0.0])
@pytest.mark.parametrize('heads,dim,vdim', [(2, 64, 128), (6, 32, 32), (2, 128, 128)])
def test_two_maps(heads, dim, vdim, softcap, start):
    cfg = T.make_config([T.attention_layer(heads=heads, kv_heads=heads // 2, dim=dim, vdim=vdim, rot_dims=dim, softcap=softcap, ff=0)])
    w = T.random_weights(cfg, 33)
    reqs, schedule = requests(GT, cfg, start)
    got = T.replay(GT.session_for(cfg, w, 'bfloat16'), reqs, schedule)
    for rid, toks in reqs.items():
        GT.check_rows(got[rid], toks, w, cfg, 'bfloat16', rid)


@pytest.mark.parametrize('start', STARTS)
@pytest.mark.parametrize('size,keep', [(0, 0), (45, 5), (130, 33)])
def test_a_window_with_kept_keys(size, keep, start):
    cfg = NC.make_config([N.attn2_layer(heads=4, kv_heads=2, dim=64, vdim=64, rot_dims=64, size=size, keep=keep, mlp=None)], width=128)
    w = NC.random_weights(cfg, 34)
    reqs, schedule = requests(N, cfg, start)
    got = T.replay(N.session_for(cfg, w, 'bfloat16'), reqs, schedule)
    for rid, toks in reqs.items():
        N.check_rows(got[rid], toks, w, cfg, 'bfloat16', rid)
