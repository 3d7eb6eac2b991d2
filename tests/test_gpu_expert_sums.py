"""A routed layer's sum formed inside the norm that reads it (expert_sum of stack_ops.hip): fewer and more experts than are requested at once, one and
two 16-byte pieces per thread, rows of few and of many tokens, the last layer's sum on the wanted rows alone, a shared expert's gated row beside
it, identities, input weights; and widths that are not taken in pieces, whose sum a launch of its own forms."""
import pytest

import narurax_cases
import rofozen_cases
import ruzinex_cases
import test_gpu_narurax
import test_gpu_rofozen
import test_gpu_ruzinex

pytestmark = pytest.mark.gpu

STEPS = [[('a', 66)], [('a', 1)], [('a', 9)], [('a', 1)]]
TOPS = [1, 4, 5, 9]


def run(mod, cases, cfg, dtype):
    toks = mod.tokens_for(cfg, sum(n for s in STEPS for _, n in s), 5)
    w = mod.weights_for(cfg, 31, dtype, toks) if hasattr(mod, 'weights_for') else cases.random_weights(cfg, 31)
    mod.check_rows(mod.replay(mod.session_for(cfg, w, dtype), {'a': toks}, STEPS)['a'], toks, w, cfg, dtype)


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('width', [70, 72, 4104])
@pytest.mark.parametrize('top', TOPS)
def test_landing_norm(top, width, dtype):
    Z = ruzinex_cases
    cfg = Z.make_config([Z.layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=Z.moe(experts=11, top=top, ff=24, shared=s)) for s in (16, 0)], width=width, vocab=61)
    run(test_gpu_ruzinex, Z, cfg, dtype)


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('top', TOPS)
def test_identities(top, dtype):
    Z = rofozen_cases
    moe = Z.moe(experts=10, identity=4, top=top, keep=2, ff=24)
    cfg = Z.make_config([Z.latent_layer(mlp=moe), Z.latent_layer(mlp=moe)], width=72)
    run(test_gpu_rofozen, Z, cfg, dtype)


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('top', TOPS)
def test_input_weights(top, dtype):
    Z = narurax_cases
    moe = Z.moe(experts=11, top=top, ff=24)
    cfg = Z.make_config([Z.attn_layer(mlp=moe), Z.attn_layer(mlp=moe)], width=72)
    run(test_gpu_narurax, Z, cfg, dtype)
