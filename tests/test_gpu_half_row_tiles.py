"""fp16 and SmoothQuant int8 products on the tiles of 128 rows of gemm_wide.hip (ids 81: 128 x 128, 82: 128 x 256): fewer K-tiles than the ring has and more, rows and columns that end
inside a tile, an odd count of tiles, scales of every kind, the fp16 residual and the SwiGLU gate.  Oracles and bounds as for the 256 x 256 tiles."""
import pytest

import test_gpu_wide_half as half
from test_gpu_wide_half import wide  # noqa: F401 (fixture)

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[81, 82], ids=['128x128', '128x256'])
def tiles(wide, request):  # noqa: F811
    wide.tllm_gemm_set_tile_cfg(request.param)
    yield wide


@pytest.mark.parametrize('sq', [True, False], ids=['int8', 'fp16'])
@pytest.mark.parametrize('k_tiles', [1, 2, 3, 4, 5, 9])
@pytest.mark.parametrize('m', [32, 127, 129, 300])
def test_product(tiles, m, k_tiles, sq):
    half.product(tiles, m, 520, k_tiles, sq)


@pytest.mark.parametrize('sq', [True, False], ids=['int8', 'fp16'])
@pytest.mark.parametrize('residual', [None, 'apart', 'in place'])
def test_several_rounds_of_tiles(tiles, residual, sq):
    half.product(tiles, 1100, 8200, 5, sq, residual=residual)


@pytest.mark.parametrize('per_channel,per_token', [(0, 0), (0, 1), (1, 0)])
def test_scales_of_a_whole_matrix(tiles, per_channel, per_token):
    half.product(tiles, 300, 520, 3, True, per_channel, per_token)


@pytest.mark.parametrize('cfg', [81, 82])
def test_swiglu_gate_of_an_fp16_prompt(wide, monkeypatch, cfg):  # noqa: F811
    monkeypatch.setattr(half, 'WIDE', cfg)
    half.test_swiglu_gate_of_an_fp16_prompt(wide)
