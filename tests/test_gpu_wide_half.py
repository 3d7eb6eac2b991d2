"""fp16 and SmoothQuant int8 products on the 256 x 256 tiles of gemm_wide.hip (id 80 of tllm_gemm_set_tile_cfg): K-tiles in every position of the
operands' rings, tiles of up to and over 128 rows, columns that end inside a tile, several rounds of tiles, scales of every kind, the fp16 residual (in
place, too) and the SwiGLU gate; the fused int8 MLP where the rule takes it.  int8 results are exact; fp16 within the bounds of test_gpu_plugins."""
import ctypes

import numpy as np
import pytest
import torch

from tensorrt_llm.plugin import capi

pytestmark = pytest.mark.gpu
WIDE = 80
MLP = (3900, 11000, 4096)                                       # rows, columns, K of the two products


class GemmParams(ctypes.Structure):
    _fields_ = [('wtype', ctypes.c_int32), ('out_dtype', ctypes.c_int32), ('M', ctypes.c_int32), ('N', ctypes.c_int32), ('K', ctypes.c_int32), ('a', ctypes.c_void_p),
                ('lda', ctypes.c_int64), ('w', ctypes.c_void_p), ('ldw', ctypes.c_int64), ('scale_col', ctypes.c_void_p), ('scale_row', ctypes.c_void_p),
                ('per_channel', ctypes.c_int32), ('per_token', ctypes.c_int32), ('c', ctypes.c_void_p), ('ldc', ctypes.c_int64)]


@pytest.fixture
def wide():
    lib = capi.load_library()
    lib.tllm_gemm.argtypes = [ctypes.POINTER(GemmParams), ctypes.c_void_p]
    lib.tllm_gemm_residual.argtypes = [ctypes.POINTER(GemmParams), ctypes.c_void_p, ctypes.c_void_p]
    lib.tllm_gemm_swiglu_quant.argtypes = [ctypes.POINTER(GemmParams)] + [ctypes.c_void_p] * 4
    lib.tllm_gemm_set_tile_cfg.argtypes = [ctypes.c_int32]
    lib.tllm_gemm_set_tile_cfg.restype = None
    lib.tllm_gemm_set_tile_cfg(WIDE)
    yield lib
    lib.tllm_gemm_set_tile_cfg(0)


def int8(*shape):
    return torch.randint(-128, 128, shape, dtype=torch.int8, device='cuda')


def product(lib, m, n, k_tiles, sq, per_channel=1, per_token=1, residual=None):
    torch.manual_seed(m + n + k_tiles)
    stream = torch.cuda.current_stream().cuda_stream
    res = (torch.randn((m, n), device='cuda') * 3).half() if residual else None
    c = res.clone() if residual == 'in place' else torch.full((m, n), 7.0, dtype=torch.float16, device='cuda')
    if sq:
        k = k_tiles * 128
        a, w = int8(m, k), int8(n, k)
        sc = torch.randint(1, 13, (n if per_channel else 1,), device='cuda').float() * 1e-4
        sr = torch.randint(1, 13, (m if per_token else 1,), device='cuda').float() * 1e-3
        q = GemmParams(3, 1, m, n, k, a.data_ptr(), k, w.data_ptr(), k, sc.data_ptr(), sr.data_ptr(), per_channel, per_token, c.data_ptr(), n)
        want = ((a.double() @ w.double().t()).float() * (sc[None, :] * sr[:, None])).half()
    else:
        k = k_tiles * 64
        a, w = torch.randn((m, k), dtype=torch.float16, device='cuda'), (torch.randn((n, k), device='cuda') / np.sqrt(k)).half()
        q = GemmParams(0, 1, m, n, k, a.data_ptr(), k, w.data_ptr(), 2 * k, None, None, 0, 0, c.data_ptr(), n)
        want = (a.double() @ w.double().t()).half()
    if residual:
        want = (want.float() + res.float()).half()
        rc = lib.tllm_gemm_residual(ctypes.byref(q), c.data_ptr() if residual == 'in place' else res.data_ptr(), stream)
    else:
        rc = lib.tllm_gemm(ctypes.byref(q), stream)
    assert rc == 0, capi.last_error()
    torch.cuda.synchronize()
    if sq:
        assert torch.equal(c, want), int((c != want).sum())
    else:
        torch.testing.assert_close(c.float(), want.float(), rtol=2e-3, atol=4e-3 if residual else 2e-3)


@pytest.mark.parametrize('sq', [True, False], ids=['int8', 'fp16'])
@pytest.mark.parametrize('k_tiles', [1, 2, 3, 4, 5, 6, 7, 13])
@pytest.mark.parametrize('m', [33, 128, 129, 300, 640])
def test_product(wide, m, k_tiles, sq):
    product(wide, m, 520, k_tiles, sq)


@pytest.mark.parametrize('sq', [True, False], ids=['int8', 'fp16'])
@pytest.mark.parametrize('residual', [None, 'apart', 'in place'])
def test_several_rounds_of_tiles(wide, residual, sq):
    """More tiles than CUs, the last ones of few rows: the next tile is requested while results leave."""
    product(wide, 2300, 16392, 5, sq, residual=residual)


@pytest.mark.parametrize('per_channel,per_token', [(0, 0), (0, 1), (1, 0)])
def test_scales_of_a_whole_matrix(wide, per_channel, per_token):
    product(wide, 300, 520, 3, True, per_channel, per_token)


def fused(lib, m, n, k, a, w1, w2, s1, s2, sr, qs):
    out = torch.full((m, n), 77, dtype=torch.int8, device='cuda')
    q = GemmParams(3, 2, m, n, k, a.data_ptr(), k, w1.data_ptr(), k, s1.data_ptr(), sr.data_ptr(), 1, 0, out.data_ptr(), n)
    assert lib.tllm_gemm_swiglu_quant(ctypes.byref(q), w2.data_ptr(), s2.data_ptr(), qs.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0, capi.last_error()
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize('k_tiles', [1, 2, 3, 4, 5, 6, 7, 13])
@pytest.mark.parametrize('m', [33, 128, 129, 300, 640])
def test_two_products_of_an_mlp(wide, m, k_tiles):
    """Against products of whole numbers, rounded to fp16 where two launches and the static quantiser round.  The kernel's exponential is another: a value of 11 bits may round the
    other way, 2^-11 of up to 127 quantised, which moves a byte by one where it lies that close to a half: 0.06 on either side at the largest, 1 byte in 100 if all of
    the 11 bits of one value in ten turn over."""
    torch.manual_seed(m + k_tiles)
    n, k = 520, 128 * k_tiles
    a, w1, w2 = int8(m, k), int8(n, k), int8(n, k)
    s1, s2 = (torch.randint(1, 13, (n,), device='cuda').float() * 2e-5 / k_tiles ** 0.5 for _ in range(2))
    sr, qs = torch.tensor([0.75], device='cuda'), torch.tensor([23.0], device='cuda')
    g, u = (((a.double() @ w.double().t()).float() * (s * sr)).half().float() for w, s in ((w1, s1), (w2, s2)))
    want = ((g / (1 + torch.exp(-g))).half().float() * u).half().float().mul(qs).round().clamp(-128, 127)
    d = (fused(wide, m, n, k, a, w1, w2, s1, s2, sr, qs).float() - want).abs()
    assert d.max() <= 1 and (d > 0).float().mean() < 1e-2 and want.unique().numel() > 100 and (want.abs() < 127).float().mean() > 0.5


def test_fused_int8_mlp(wide):
    """Rows, columns and K for which the rule takes these tiles (test_stack_host_runtime.py): the same bytes as by the one-tile-per-workgroup form."""
    torch.manual_seed(5)
    m, n, k = MLP
    a, w1, w2 = int8(m, k), int8(n, k), int8(n, k)
    s1, s2 = (torch.randint(1, 13, (n,), device='cuda').float() * 2e-6 for _ in range(2))
    sr, qs = torch.tensor([0.75], device='cuda'), torch.tensor([23.0], device='cuda')
    got = []
    for cfg in (0, -2):
        wide.tllm_gemm_set_tile_cfg(cfg)
        got.append(fused(wide, m, n, k, a, w1, w2, s1, s2, sr, qs))
    assert torch.equal(*got) and got[0].unique().numel() > 100


def test_swiglu_gate_of_an_fp16_prompt(wide):
    """A session's prompt by these tiles against the same by 128 x 128 ones."""
    from tensorrt_llm.runtime.native import NativeSession
    D, I, V, L = 256, 704, 512, 2
    g = torch.Generator(device='cuda').manual_seed(3)
    r = lambda *s: (torch.randn(s, generator=g, device='cuda') * s[-1] ** -0.5).half()
    t = {'vocab_embedding.weight': r(V, D) * 16, 'ln_f.weight': torch.ones(D, dtype=torch.float16, device='cuda'), 'lm_head.weight': r(V, D)}
    for i in range(L):
        p = 'layers.%d.' % i
        for name in ('input_layernorm', 'post_layernorm'):
            t[p + name + '.weight'] = torch.ones(D, dtype=torch.float16, device='cuda')
        for name, n, k in (('attention.qkv', 3 * D, D), ('attention.dense', D, D), ('mlp.fc', I, D), ('mlp.gate', I, D), ('mlp.proj', D, I)):
            t[p + name + '.weight'] = r(n, k)
    ids = np.random.default_rng(4).integers(3, V, (2, 70)).astype(np.int32)
    lens, logits = np.array([70, 70], np.int32), []
    for cfg in (WIDE, 8):
        wide.tllm_gemm_set_tile_cfg(cfg)
        s = NativeSession(dict(num_layers=L, num_heads=2, hidden_size=D, inter_size=I, vocab_size=V, max_position_embeddings=128, rms_norm_eps=1e-6, quant_mode=0))
        for name, x in t.items():
            s.set_tensor(name, x)
        torch.cuda.synchronize()
        s.finalize()
        s.setup(2, 70, 1)
        s.context(ids, lens)
        logits.append(s.logits().astype(np.float64))
        s.close()
    assert np.linalg.norm(logits[0] - logits[1]) < 4e-3 * np.linalg.norm(logits[1]) and np.isfinite(logits[0]).all()
