"""Grouped products of few rows (slim_group_kernel and the stream form's shapes for groups, gemm_slim_impl.h): on both sides of the lines between them in
rows (8), products and length of a row; every group with all of a step's rows, in one and two row tiles, and groups with none, one or several; rows of W that
end inside a block and columns that end inside a workgroup.  Bounds as in the designs' own tests."""
import pytest

import ruzinex_cases as Z
import test_gpu_ruzinex as R

pytestmark = pytest.mark.gpu

ROWS = [2, 8, 9, 16, 17, 31]


@pytest.mark.parametrize('width', [72, 512, 1032, 2056])
@pytest.mark.parametrize('experts,top,ff', [(32, 32, 524), (40, 3, 690), (32, 32, 128)])
def test_steps_of_few_tokens(experts, top, ff, width):
    cfg = Z.make_config([Z.layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=Z.moe(experts=experts, top=top, ff=ff - ff % 8, shared=0))], width=width, vocab=61)
    reqs = {m: R.tokens_for(cfg, m, 50 + m) for m in ROWS}
    w = R.weights_for(cfg, 98, 'bfloat16', reqs)
    got = R.replay(R.session_for(cfg, w, 'bfloat16', max_sequences=len(ROWS)), reqs, [[(m, m)] for m in ROWS])
    for m, toks in reqs.items():
        R.check_rows(got[m], toks, w, cfg, 'bfloat16', f'{m} rows')
