"""Decode products of several rows (gemv_impl.h), whose activation rows come all at once up to K = 4096 and one after the other beyond: row by row the bits of the same call
on one row, in every weight type, with each prologue, and with fewer rows than the form holds.  (As many columns as keep one row off the form that splits K.)"""
import ctypes

import numpy as np
import pytest
import torch

from tensorrt_llm.plugin import capi
from test_gpu_plugins import _GemvParams

pytestmark = pytest.mark.gpu
FP16, WOQ8, WOQ4, SQ = range(4)
COLUMNS = 8200
K_BYTES = {FP16: 2, WOQ8: 1, WOQ4: 0.5, SQ: 1}


@pytest.mark.parametrize('k', [32, 2080, 4096, 4128])
@pytest.mark.parametrize('wtype,pro', [(FP16, 0), (FP16, 1), (WOQ8, 0), (WOQ8, 1), (WOQ4, 0), (WOQ4, 1), (SQ, 0), (SQ, 2), (SQ, 3), (SQ, 4), (SQ, 5)])
def test_rows_together_are_the_rows_alone(wtype, pro, k):
    lib = capi.load_library()
    lib.tllm_gemv.argtypes = [ctypes.POINTER(_GemvParams), ctypes.c_void_p]
    lib.tllm_gemv.restype = ctypes.c_int32
    lib.tllm_gemv_set_mfma_rows.argtypes = [ctypes.c_int32]
    lib.tllm_gemv_set_mfma_rows.restype = None
    g = torch.Generator(device='cuda').manual_seed(k + 10 * pro + wtype)
    ldw = (int(k * K_BYTES[wtype]) + 15) // 16 * 16
    if wtype == FP16:
        w = (torch.randn((COLUMNS, k), device='cuda', generator=g) / k ** 0.5).half()
    else:
        w = torch.randint(-128, 128, (COLUMNS, ldw), dtype=torch.int8, device='cuda', generator=g)
    scale = torch.rand(COLUMNS, device='cuda', generator=g) * 2e-3 + 1e-4
    scale = scale.half() if wtype in (WOQ8, WOQ4) else scale.float()
    x = torch.randint(-127, 128, (8, k), dtype=torch.int8, device='cuda', generator=g) if wtype == SQ and pro == 0 else torch.randn((8, k), device='cuda', generator=g).half()
    gamma = (torch.rand(k, device='cuda', generator=g) + 0.5).half()
    act, row_scale, dynamic = torch.tensor([37.0], device='cuda'), torch.tensor([0.013], device='cuda'), torch.zeros(8, device='cuda')

    def product(first, m):
        y = torch.full((m, COLUMNS), 7.0, dtype=torch.float16, device='cuda')
        q = _GemvParams(wtype, pro, 0, 1, m, COLUMNS, k, x[first:].data_ptr(), k, w.data_ptr(), ldw, scale.data_ptr() if wtype != FP16 else None,
                        row_scale.data_ptr() if wtype == SQ else None, 1, 0, gamma.data_ptr(), 1e-6, act.data_ptr(), dynamic.data_ptr(), None, None, None, y.data_ptr(), COLUMNS)
        assert lib.tllm_gemv(ctypes.byref(q), torch.cuda.current_stream().cuda_stream) == 0, capi.last_error()
        torch.cuda.synchronize()
        return y.cpu().numpy()

    lib.tllm_gemv_set_mfma_rows(0)  # (several int8 rows stay with the form under test)
    try:
        alone = np.concatenate([product(m, 1) for m in range(8)])
        assert np.abs(alone.astype(np.float64)).max() > 0.01 and np.isfinite(alone).all()
        for m in (2, 3, 4, 5, 8):
            np.testing.assert_array_equal(product(0, m), alone[:m], err_msg=f'{m} rows')
    finally:
        lib.tllm_gemv_set_mfma_rows(-1)
