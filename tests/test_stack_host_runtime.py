"""Host side of the stack engine's step - scratch, pinned memory, launch shapes - over a stand-in for the HIP runtime (hip_stub.cpp), without a
GPU: nothing is computed, but every allocation and launch is the real code's.  Each scenario runs in a process of its own, with the stand-in
loaded ahead of the library."""
import ctypes
import os
import re
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope='module')
def stub(tmp_path_factory):
    out = str(tmp_path_factory.mktemp('stub') / 'hip_stub.so')
    subprocess.run(['g++', '-shared', '-fPIC', '-std=c++17', '-O1', '-D__HIP_PLATFORM_AMD__', '-I/opt/rocm/include', os.path.join(HERE, 'hip_stub.cpp'), '-o', out],
                   check=True)
    return out


def run(stub, scenario, *args):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), stub, scenario, *map(str, args)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


# ------------------------------------------------------------------------------------------------------------ in the child process
class Stub:
    def __init__(self, path):
        self.lib = ctypes.CDLL(path, mode=ctypes.RTLD_GLOBAL)
        self.lib.stub_budget.argtypes = self.lib.stub_has_allocation.argtypes = [ctypes.c_size_t]
        self.lib.stub_live.restype = self.lib.stub_largest.restype = self.lib.stub_pinned_bytes.restype = ctypes.c_size_t
        self.lib.stub_launched.restype = ctypes.c_char_p
        for p in (os.path.dirname(HERE), os.path.join(os.path.dirname(HERE), 'trtllm-llama_amd'), HERE):
            sys.path.insert(0, p)

    def __getattr__(self, name):
        return getattr(self.lib, 'stub_' + name)

    def kernels(self):
        return self.launched().decode().split()


def engine(cfg, cases, dtype='bfloat16', **kw):
    from tensorrt_llm.runtime import RaggedGenerationSession
    return RaggedGenerationSession(cases.as_model(cfg, cases.random_weights(cfg, 1)), dtype=dtype, **kw)


def step(s, rid, n, want=1, **kw):
    return s.step([(rid, [1] * n, list(range(want)))], end=(rid,), **kw)


def chunk_floats(tokens, entries, heads, vector_heads, dim, vectors, mamba=False):
    """Per chunk of 16 rows: `vectors` of them per row and head (Mamba-2: per group), a 16 x 16 matrix per head (delta rule: two) and the decays over
    the chunk (Mamba-2: 48 numbers)."""
    chunks = tokens // 16 + entries + 1
    return chunks * (vectors * 16 * dim * vector_heads + heads * (256 * (vectors - 1) + (48 if mamba else dim)))


def scratch_of_the_state_layers(stub):
    """What the chunked recurrences keep is what is allocated: Mamba-2's vectors once per group, not per head."""
    import narurax_cases as N
    import rofozen_cases as M
    import tolenex_cases as H
    for cases, layer, size in ((M, M.mamba_layer(heads=64, vdim=16, state=128, groups=8), (64, 8, 128, 2)),
                               (M, M.mamba_layer(heads=6, vdim=16, state=64, groups=6), (6, 6, 64, 2)),
                               (N, N.delta_layer(heads=8, kv_heads=2, dim=128, vdim=64), (8, 8, 128, 3)),
                               (H, H.hgrn2_layer(heads=4, dim=192, vdim=32), (4, 4, 192, 2))):
        s = engine(cases.make_config([layer]), cases, max_tokens=2048, max_sequences=4)
        stub.forget()
        step(s, 'a', 2000)
        assert any('chunk_walk_kernel' in k for k in stub.kernels())
        heads, vector_heads, dim, vectors = size
        floats = chunk_floats(2000, 4, heads, vector_heads, dim, vectors, mamba=cases is M)
        assert stub.has_allocation(4 * floats), (layer, 4 * floats)


def scratch_that_leaves_room(stub):
    """With the last free bytes short of the state layers' scratch, a step still has its mandatory buffers, and walks row by row."""
    import narurax_cases as N
    cfg = N.make_config([N.delta_layer(heads=8, kv_heads=2, dim=128, vdim=64)])
    s = engine(cfg, N, max_tokens=2048, max_sequences=4)
    before = stub.live()
    step(s, 'a', 1024)
    need, floats = stub.live() - before, chunk_floats(1024, 4, 8, 8, 128, 3)
    assert any('chunk_walk_kernel' in k for k in stub.kernels())
    for spare in (floats // 16, 2 * floats, 4 * floats - 4096):
        s = engine(cfg, N, max_tokens=2048, max_sequences=4)
        stub.budget(stub.live() + need - 4 * floats + spare)
        stub.forget()
        step(s, 'a', 1024)
        assert stub.kernels() and not any('chunk_walk_kernel' in k for k in stub.kernels())
        stub.budget(2 ** 64 - 1)


def step_behind_one_that_found_no_memory(stub):
    """A step that fails for want of memory gives its scratch back; a smaller one behind it makes its own."""
    import narurax_cases as N
    cfg = N.make_config([N.delta_layer(heads=8, kv_heads=2, dim=128, vdim=64)])
    s = engine(cfg, N, max_tokens=2048, max_sequences=4)
    step(s, 'a', 100)
    stub.budget(stub.live() + (64 << 10))
    try:
        step(s, 'b', 1500)
    except RuntimeError as e:
        assert 'out of memory' in str(e)
    else:
        raise AssertionError('the budget holds the step')
    stub.budget(2 ** 64 - 1)
    stub.forget()
    step(s, 'c', 20)
    assert stub.kernels()


def pinned_rows(stub):
    """Requests come in one by one: the pinned room for wanted rows grows by doubling, up to 8 MiB of logits, and nothing is pinned for rows that
    go to nobody."""
    import rofozen_cases as M
    cfg = M.make_config([M.mamba_layer(heads=2, vdim=8, state=16, groups=1)], vocab=32000)
    s = engine(cfg, M, max_tokens=2048, max_sequences=4)
    step(s, 0, 70, 0)  # (the step's scratch and its pinned metadata are made here)
    lib, none = s.engine._h, stub.host_mallocs()
    import tensorrt_llm.runtime.stack as stack
    one, pos, slot, table = (np.array(v, np.int32) for v in ([3], [0], [0], [[0]]))
    b = stack.Batch(1, 1, 1, 1, one.ctypes.data, (count := np.array([1], np.int32)).ctypes.data, pos.ctypes.data, slot.ctypes.data, table.ctypes.data, pos.ctypes.data)
    assert stack.load_library().tllm_stack_step(lib, ctypes.byref(b), None, None, None) == 0
    assert stub.host_mallocs() == none
    step(s, 1, 70, 70)  # (rows by copy; the scratch for the most rows)
    scratch = stub.host_mallocs()
    for n in range(1, 66):
        logits, ids = step(s, n + 1, 70, n)
        assert logits.shape == (n, 32000) and 'deliver_kernel' in stub.launched().decode()
    assert stub.host_mallocs() - scratch == 8  # 1, 2, 4, ... 64 and 65 rows
    assert stub.pinned_bytes() <= (8 << 20) + 65 * 64 * 8 + (64 << 10)


def streams_in_turn(stub):
    """A step behind one that returned with its rows, on another stream, waits for nothing else on the device."""
    import rofozen_cases as M
    s = engine(M.make_config([M.mamba_layer(heads=2, vdim=8, state=16, groups=1)]), M, max_tokens=64, max_sequences=1)
    take = s.engine.step
    s.step([('a', [1], [0])])  # (makes its scratch)
    syncs = stub.device_syncs()
    for stream in (0, 64, 64, 128, 0):
        s.engine.step = lambda *a, **k: take(*a, **dict(k, stream=stream))
        s.step([('a', [1], [0])])
    assert stub.device_syncs() == syncs


def who_waits(stub):
    """The host watches for a step's rows unless the step's products alone take longer than it would: of 2 ms at 1.31 PFLOP/s in bfloat16, 0.15 in fp32."""
    import ruzinex_cases as Z

    class Zeros:  # (nothing is computed)
        standard_normal = staticmethod(lambda shape: np.zeros(shape, np.float32))
    np.random.default_rng = lambda seed: Zeros
    for dtype, rate in (('bfloat16', 1.31e15), ('float32', 0.15e15)):
        width, ff, d = 1024, 6144, 32
        s = engine(Z.make_config([Z.layer(heads=2, kv_heads=1, dim=d, vdim=d, mlp=Z.dense(ff=ff))], width=width, vocab=64), Z, dtype=dtype, max_tokens=140000, max_batch_tokens=140000, max_sequences=1)
        edge = 2e-3 * rate / (2 * width * (3 * ff + 6 * d))
        for tokens, watches in ((1, True), (int(0.98 * edge), True), (int(1.02 * edge), False)):
            before = stub.stream_syncs()
            step(s, 'a', tokens)
            assert stub.stream_syncs() - before == (0 if watches else 1), (dtype, tokens)


def rows_to_the_edge(stub):
    """The caller's rows begin and end at the edge of what may be written, whatever their size; a step of that many rows stays within them."""
    import mmap
    import rofozen_cases as M
    import tensorrt_llm.runtime.stack as stack
    libc = ctypes.CDLL(None)
    for vocab in (16, 1024, 1027, 32000):
        s = engine(M.make_config([M.mamba_layer(heads=2, vdim=8, state=16, groups=1)], vocab=vocab), M, max_tokens=256, max_sequences=4)
        tokens, zero, one, wanted = np.ones(3, np.int32), np.zeros(4, np.int32), np.full(1, 3, np.int32), np.arange(3, dtype=np.int32)
        for want in (1, 3):
            n, page = want * vocab * 4, mmap.PAGESIZE
            pages = -(-n // page)
            m = mmap.mmap(-1, (pages + 2) * page)
            base = ctypes.addressof(ctypes.c_char.from_buffer(m))
            for closed in (base, base + (pages + 1) * page):
                assert libc.mprotect(ctypes.c_void_p(closed), page, 0) == 0
            for at in (base + page, base + (pages + 1) * page - n):
                b = stack.Batch(3, 1, want, 1, tokens.ctypes.data, one.ctypes.data, zero.ctypes.data, zero.ctypes.data, zero.ctypes.data,
                                wanted.ctypes.data)
                stub.forget()
                assert stack.load_library().tllm_stack_step(s.engine._h, ctypes.byref(b), at, None, None) == 0
                assert any('deliver' in k for k in stub.kernels())


def huge_step(stub):
    """One prompt of 131072 tokens beside 300 decoded ones, 64 heads: tiles x entries x heads of one launch are more than a grid's x dimension takes."""
    import ruzinex_cases as Z
    cfg = Z.make_config([Z.layer(heads=64, kv_heads=8, dim=64, vdim=64, rot_dims=32)], width=64)
    s = engine(cfg, Z, max_tokens=160000, max_sequences=301)
    for i in range(300):
        s.step([(i, [1], [0])])
    stub.forget()
    s.step([('long', [1] * 131072, [0])] + [(i, [1], [0]) for i in range(300)])
    assert any('attn_prefill_kernel' in k for k in stub.kernels())
    s.step([('long', [1] * 40, [0])] + [(i, [1], [0]) for i in range(300)])
    assert any('attn_prompt_kernel' in k for k in stub.kernels())


def many_small_rows(stub):
    """More wanted rows of a small vocabulary than a grid has in y."""
    import rofozen_cases as M
    cfg = M.make_config([M.mamba_layer(heads=2, vdim=8, state=16, groups=1)], vocab=16, width=32)
    s = engine(cfg, M, max_tokens=80000, max_sequences=1)
    logits, ids = step(s, 'a', 70000, 70000)
    assert logits.shape == (70000, 16) and ids.shape == (70000,)


def tile_shapes(stub):
    """The sizes of test_gpu_product_tiles.py take the tile shapes they are listed under."""
    import test_gpu_product_tiles as P
    import ruzinex_cases as Z
    import tolenex_cases as T

    def shapes(cfg, cases, rows, want=1):
        s = engine(cfg, cases, max_tokens=2048, max_sequences=1)
        stub.forget()
        step(s, 'a', rows, want)
        found = [re.search(r'gemm_glds_kernelILi\d+ELi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)', k) for k in stub.kernels()]
        return [(32 * int(m[1]) * int(m[3]), 32 * int(m[2]) * int(m[4])) for m in found if m]

    for shape, (columns, ff, grouped) in P.SHAPES.items():
        for c in (columns, columns - 1):
            assert shapes(P.plain_config(c, 64), Z, P.ROWS, P.ROWS)[-1] == shape, (shape, c)
        assert shapes(P.gated_config(Z.dense(ff=ff), 64), Z, P.ROWS)[2] == shape, (shape, ff)
        assert shapes(P.gated_config(Z.moe(experts=2, top=2, ff=grouped, shared=0), 64), Z, P.ROWS)[3] == shape, (shape, grouped)
    for shape, (experts, top) in P.FEW.items():
        assert shapes(P.gated_config(Z.moe(experts=experts, top=top, ff=192, shared=0), 64), Z, P.ROWS)[-2:] == [shape] * 2, shape
    for shape, (rows, width) in P.RESIDUAL.items():
        assert [x for x in shapes(P.residual_config(width), T, rows)][1::2] == [shape] * 2, shape


def wide_tiles(stub):
    """The sizes of test_gpu_wide_tiles.py take the 256 x 256 tiles of gemm_wide_impl.h: (ways out of wide::Out, grouped) of a step's products."""
    import ruzinex_cases as Z
    import sodudra_cases as S
    import test_gpu_product_tiles as P
    import test_gpu_wide_tiles as G
    import tolenex_cases as T

    class Zeros:  # (nothing is computed)
        standard_normal = uniform = staticmethod(lambda *a, size=None, **k: np.zeros(size if size is not None else a[-1], np.float32))
    np.random.default_rng = lambda seed: Zeros
    for cases in (S, T, Z):
        cases.bf16_round = lambda x: x
    store, gated, fp32, resid, resid_gate = range(5)

    def outs(cfg, cases, *steps):
        s = engine(cfg, cases, max_tokens=4096, max_batch_tokens=4096, max_sequences=1)
        for rows, want in steps:
            stub.forget()
            step(s, 'a', rows, want)
            found = [re.search(r'wide_kernelILi\d+ELi(\d+)ELb([01])', k) for k in stub.kernels()]
            yield {(int(m[1]), int(m[2])) for m in found if m}

    for k in sorted({k for _, k in G.PLAIN}):
        for found in outs(P.plain_config(G.COLUMNS, k), Z, *((rows, rows) for rows, at in G.PLAIN if at == k)):
            assert (fp32, 0) in found, k
    rows, k = G.PLAIN[0]
    assert not next(outs(P.plain_config(G.COLUMNS - 1, k), Z, (rows, rows)))
    assert (gated, 0) in next(outs(G.gated_config(), Z, (G.GATED[0], 1)))
    for tokens, *sizes in G.GROUPED:
        assert (gated, 1) in next(outs(G.grouped_config(*sizes), Z, (tokens, 1))), sizes
    assert (fp32, 1) in next(outs(G.grouped_config(*G.GROUPED[-1][1:]), Z, (G.GROUPED[-1][0], 1)))
    assert (resid_gate, 0) in next(outs(G.residual_config(T), T, (G.RESIDUAL[0], 1)))
    assert (resid, 0) in next(outs(G.residual_config(S), S, (G.RESIDUAL[0], 1)))


def row_tiles(stub):
    """The sizes of test_gpu_row_tiles.py take the tiles of gemm_wide_impl.h that they are listed under."""
    import ruzinex_cases as Z
    import sodudra_cases as S
    import test_gpu_product_tiles as P
    import test_gpu_row_tiles as G
    import tolenex_cases as T

    class Zeros:  # (nothing is computed)
        standard_normal = uniform = staticmethod(lambda *a, size=None, **k: np.zeros(size if size is not None else a[-1], np.float32))
    np.random.default_rng = lambda seed: Zeros
    for cases in (S, T, Z):
        cases.bf16_round = lambda x: x
    store, gated, fp32, resid, resid_gate = range(5)

    def tiles(cfg, cases, rows, want=1):
        s = engine(cfg, cases, max_tokens=2048, max_sequences=1)
        stub.forget()
        step(s, 'a', rows, want)
        found = [re.search(r'4wide\d+gemm_glds_kernelILi\d+ELi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)ELi\d+ELi(\d+)', k) for k in stub.kernels()]
        return [(32 * int(m[1]) * int(m[3]), 32 * int(m[2]) * int(m[4]), int(m[5])) for m in found if m]

    for shape, columns in G.COLUMNS.items():
        assert tiles(P.plain_config(columns, 64), Z, P.ROWS, P.ROWS)[-1] == (*shape, fp32)
        assert (*shape, gated) in tiles(G.shared_config(G.SHARED[shape]), Z, P.ROWS), shape
    s = engine(G.shared_config(*G.WIDE_SHARED), Z, max_tokens=2048, max_sequences=1)
    stub.forget()
    step(s, 'a', P.ROWS, 1)
    assert any(f'wide_kernelILi4ELi{gated}ELb0' in k for k in stub.kernels())
    for shape, (rows, width) in G.RESIDUAL.items():
        assert (*shape, resid) in tiles(G.residual_config(width), S, rows), shape
        assert (*shape, resid_gate) in tiles(P.residual_config(width), T, rows), shape


def convolution_of_single_rows(stub):
    """A step of one row per entry has no launch for a convolution of 4 taps, whatever the layers of test_gpu_conv_step.py; other steps and other taps do."""
    import test_gpu_conv_step as G
    import narurax_cases as N
    import rofozen_cases as M
    for name, layer in G.LAYERS.items():
        cases = N if name.startswith('delta') else M
        for taps in (4, 3):
            layer['mixer']['conv'] = taps
            s = engine(cases.make_config([layer]), cases, max_tokens=64, max_sequences=2)
            for rows in (5, 1, 1, 2):
                stub.forget()
                step(s, 'a', rows)
                kernels = stub.kernels()
                assert any('ssm_conv' in k for k in kernels) == (rows > 1 or taps != 4), (name, taps, rows)
                assert any(re.search(r'(ssm|delta)_step_kernelILi7ELb1', k) for k in kernels) == (rows == 1 and taps == 4), (name, taps, rows)


def in_lone_steps(stub, pattern, cfg, cases, dtype='bfloat16', rows=1):
    """-> matches of `pattern` among the kernels of a step of `rows` tokens behind a prompt."""
    s = engine(cfg, cases, dtype, max_tokens=64, max_sequences=1)
    s.step([('a', [1, 2, 3], [0])])
    stub.forget()
    s.step([('a', [1] * rows, [0])])
    return [m for m in (re.search(pattern, k) for k in stub.kernels()) if m]


def lone_norms(stub):
    """A lone token's rows are normed by their readers at the sizes that test_gpu_lone_norm.py and test_gpu_lone_out_norm.py list for it, and not just outside."""
    import rofozen_cases as F
    import tolenex_cases as T

    class Zeros:  # (nothing is computed)
        standard_normal = staticmethod(lambda shape: np.zeros(shape, np.float32))
        uniform = staticmethod(lambda lo, hi, size=None: np.full(size, lo, np.float32))
    np.random.default_rng = lambda seed: Zeros
    row_norm = r'row_norm_kernelILi\d+ELi\d+ELi\d+ELi(\d+)E'
    mamba = dict(heads=2, vdim=12, state=16, groups=1, norm_groups=1)  # (rows of 24: their own norm has a launch)
    for width in (16, 96, 104, 512, 528, 1024, 1040, 2048, 2064, 4096, 4112):
        served = width % 16 == 0 and width <= 4096
        cfg = F.make_config([F.mamba_layer(mlp=F.dense(ff=40), **mamba), F.latent_layer(mlp=F.moe(experts=4, identity=2, top=2, count=1, keep=1))], width=width)
        assert [m[1] for m in in_lone_steps(stub, row_norm, cfg, F)] == ['0'] * 3 * served, width  # two mixers' first products and a feed-forward's
        assert len(in_lone_steps(stub, 'moe_logits_norm_kernel', cfg, F)) == served, width
        assert not in_lone_steps(stub, 'row_norm|logits_norm', cfg, F, 'float32') and not in_lone_steps(stub, 'row_norm|logits_norm', cfg, F, rows=2)
    for width, parts, served in ((96, 1, 1), (96, 2, 1), (96, 4, 1), (96, 3, 0), (1040, 2, 1), (1040, 4, 1), (2048, 4, 1), (4096, 1, 1), (4096, 4, 1), (4112, 4, 0), (1024, 8, 0), (2048, 8, 1), (4096, 8, 1)):
        cfg = T.make_config([T.attention_layer(heads=2, kv_heads=1, dim=16, vdim=16, rot_dims=8, ff=40)], width=width, groups=parts)
        assert [m[1] for m in in_lone_steps(stub, row_norm, cfg, T)] == [str(parts)] * served, (width, parts)
    for heads, vdim, parts, served in ((2, 8, 1, 1), (4, 16, 4, 1), (4, 18, 4, 0), (6, 16, 3, 0), (8, 64, 8, 0), (32, 64, 1, 1), (32, 64, 8, 1), (32, 96, 8, 0), (64, 64, 4, 1), (64, 64, 8, 1), (64, 66, 8, 0)):
        cfg = F.make_config([F.mamba_layer(heads=heads, vdim=vdim, state=8, groups=1, norm_groups=parts)], width=100)  # (the layer's own rows are no whole pieces)
        assert [m[1] for m in in_lone_steps(stub, row_norm, cfg, F)] == [str(parts)] * served, (heads, vdim, parts)


def shifts_and_starts(stub):
    """The token shift inside its norm's launch, and the start of a step in one, at the sizes of test_gpu_shift_step.py and test_gpu_step_start.py."""
    import narurax_cases as N
    delta = dict(heads=2, kv_heads=1, dim=8, vdim=8)
    for width in (96, 98, 260, 4096, 4100, 8192, 8196):
        cfg = N.make_config([N.delta_layer(**delta)] * 2, width=width)
        for dtype in ('bfloat16', 'float32'):
            together = width % 4 == 0 and width <= 8192
            assert len(in_lone_steps(stub, r'hyper_norm_vec_kernelILi\d+ELi1ELi\d+ELb1', cfg, N, dtype)) == 2 * together, (width, dtype)
            assert len(in_lone_steps(stub, 'token_shift_kernel', cfg, N, dtype)) == 2 * (not together), (width, dtype)
            assert len(in_lone_steps(stub, 'token_shift_kernel', cfg, N, dtype, rows=2)) == 2
    for width in (8, 96, 100, 2056):
        cfg = N.make_config([N.delta_layer(**delta)], width=width)
        for rows in (1, 16, 17):
            one = width % 8 == 0 and rows <= 16
            assert [len(in_lone_steps(stub, name, cfg, N, rows=rows)) for name in ('begin_kernel', 'fetch_kernel', 'embed')] == ([1, 0, 0] if one else [0, 1, 2]), (width, rows)


def packed_prompts(stub):
    """Batches of test_gpu_ragged_prompts.py that leave their padding rows out, and such that do not; products of either have a kernel that was chosen by measuring."""
    import test_gpu_ragged_prompts as G
    from tensorrt_llm.plugin import capi
    lib = capi.load_library()
    lib.tllm_gemm_tactic_lookup.restype = ctypes.c_int32
    for mode, wtype in (('fp16', 0), ('sq_static_pc', 3)):
        _, session = G.sessions(mode, 1)
        s = session(4, G.S)
        for lens in G.BATCHES:
            stub.forget()
            s.context(np.zeros((4, G.S), np.int32), np.array(lens, np.int32))
            assert any('gather_rows' in k for k in stub.kernels()) == (sum(lens) <= 1232), (mode, lens)
        s.close()
        lib.tllm_gemm_tactics_clear()
        for prompt, packed in ((330, 1000), (G.S, 1024), (G.S, 1232)):
            s = session(4, prompt)
            assert lib.tllm_gemm_tactic_lookup(wtype, 4 * prompt, 6144, 2048) > 0 and lib.tllm_gemm_tactic_lookup(wtype, packed, 6144, 2048) > 0, (mode, prompt, packed)
            s.close()
            lib.tllm_gemm_tactics_clear()


def two_int8_products(stub):
    """The sizes of test_gpu_wide_half.py's MLP take the tiles of gemm_wide.hip by their cost, or by their id; the one-tile form and small ones do not."""
    import test_gpu_wide_half as G
    from tensorrt_llm.plugin import capi
    lib = capi.load_library()
    lib.tllm_gemm_swiglu_quant.argtypes = [ctypes.POINTER(G.GemmParams)] + [ctypes.c_void_p] * 4
    for cfg, (m, n, k), wide in ((0, G.MLP, True), (-2, G.MLP, False), (0, (300, 520, 384), False), (G.WIDE, (300, 520, 384), True)):
        lib.tllm_gemm_set_tile_cfg(0)
        lib.tllm_gemm_set_tile_cfg(cfg)
        stub.forget()
        q = G.GemmParams(3, 2, m, n, k, 4096, k, 4096, k, 4096, 4096, 1, 0, 4096, n)
        assert lib.tllm_gemm_swiglu_quant(ctypes.byref(q), 4096, 4096, 4096, None) == 0
        assert [bool(re.search('wide_kernelILi3ELi6', x)) for x in stub.kernels()] == [wide], (cfg, m)


def int8_products(stub):
    """SmoothQuant products without a measured choice: the tiles of 128 rows where they save a round or fit better, 256 x 128 at equal counts, one round of 256 x 256 rather than two of 128 x 256."""
    import test_gpu_wide_half as G
    from tensorrt_llm.plugin import capi
    lib = capi.load_library()
    lib.tllm_gemm.argtypes = [ctypes.POINTER(G.GemmParams), ctypes.c_void_p]
    for m, n, k, want in ((384, 13824, 5120, 'gemm_sqp'), (512, 11008, 4096, 'gemm_sqp'), (1024, 5120, 5120, 'gemm_sqp'), (2500, 5504, 2048, 'wide_kernelILi3E'), (2500, 6144, 2048, 'wide_kernelILi3E'),
                          (640, 11008, 4096, 'wide16gemm_glds_kernelILi3ELi2ELi4ELi2ELi2E'), (1400, 11008, 4096, 'wide16gemm_glds_kernelILi3ELi2ELi4ELi2ELi2E'),
                          (512, 4096, 4096, 'wide16gemm_glds_kernelILi3ELi2ELi4ELi2ELi1E'), (1024, 4096, 4096, 'wide16gemm_glds_kernelILi3ELi2ELi4ELi2ELi1E')):
        stub.forget()
        q = G.GemmParams(3, 1, m, n, k, 4096, k, 4096, k, 4096, 4096, 1, 0, 4096, n)
        assert lib.tllm_gemm(ctypes.byref(q), None) == 0
        assert want in stub.kernels()[-1], (m, n, k, stub.kernels())


def cold_weights(stub):
    """Products are timed on weights that rotate through more than the last-level cache, small ones too; with little memory free on fewer, and are chosen all the same."""
    from tensorrt_llm.plugin import capi
    lib = capi.load_library()
    lib.tllm_gemm_profile.argtypes = [ctypes.c_int32] * 4 + [ctypes.c_void_p] * 3
    largest = 0
    for wtype, n, k in ((0, 64, 64), (3, 2752, 1024), (0, 1024, 1024), (0, 4096, 4096)):
        for budget in (2 ** 64 - 1, 64 << 20):
            lib.tllm_gemm_tactics_clear()
            stub.budget(budget)
            assert lib.tllm_gemm_profile(wtype, 128, n, k, None, None, None) == 0 and lib.tllm_gemm_tactic_lookup(wtype, 128, n, k) > 0, (wtype, n, k)
            stub.budget(2 ** 64 - 1)
            largest = max(largest, n * k * (2 if wtype == 0 else 1))
        assert (384 << 20) - largest <= stub.largest() <= (384 << 20) + 16, (n, k, stub.largest())


def low_rank_pairs(stub):
    """A delta layer's two low-rank pairs are one product of two where one launch serves it; rows of tiles that end inside a stage of 64 go one by one, not by the
    register-staged tiles."""
    import narurax_cases as N
    from tensorrt_llm.runtime import RaggedGenerationSession
    for rank in (8, 40, 64, 72, 96, 128):
        cfg = N.make_config([N.delta_layer(heads=2, kv_heads=1, dim=96, vdim=96)], width=256)
        s = RaggedGenerationSession(N.as_model(cfg, N.random_weights(cfg, 1, ranks=(rank, rank))), dtype='bfloat16', max_tokens=256, max_sequences=1)
        for rows in (1, 8, 31, 32, 40):
            stub.forget()
            step(s, 'a', rows)
            kernels = stub.kernels()
            first = next(i for i, k in enumerate(kernels) if 'token_shift' in k or re.search(r'hyper_norm_vec_kernelILi7ELi1ELi1ELb1', k)) + 1  # the mixer's first product
            last = next(i for i, k in enumerate(kernels) if re.search(r'delta_(scan|step)', k))
            found = [k for k in kernels[first + 1:last] if 'conv' not in k]
            if rows < 32 or rank % 64 == 0:
                assert len(found) == 1, (rank, rows, found)
            elif rank > 64:
                assert [bool(re.search('gemm_glds', k)) for k in found] == [True, False] * 2 and all('fma_tile' in k for k in found[1::2]), (rank, rows, found)


def norms_without_a_sum(stub):
    """A norm of any number of streams carries the code of the experts' sum only where there is one to form."""
    import narurax_cases as N
    import ruzinex_cases as Z
    import vetipel_cases as V

    def summing(cfg, cases):
        s = engine(cfg, cases, max_tokens=256, max_sequences=1)
        stub.forget()
        step(s, 'a', 40)
        found = [re.search(r'(?:hyper_norm|land)_vec_kernelI.*Lb([01])E', k) for k in stub.kernels()]
        assert any(found)
        return {m[1] for m in found if m}

    for width in (96, 4104):
        for streams in (1, 2, 3, 8):
            assert summing(V.make_config([V.window_layer()] * 2, width=width, streams=streams), V) == {'0'}, (width, streams)
        assert summing(Z.make_config([Z.layer(mlp=Z.dense(ff=24))], width=width), Z) == {'0'}
        for cases, layer in ((N, N.attn_layer(mlp=N.moe())), (Z, Z.layer(mlp=Z.moe()))):
            assert summing(cases.make_config([layer] * 2, width=width), cases) == {'0', '1'}, (width, cases)


def few_row_forms(stub):
    """Products of 2 .. 31 rows take the form that their rows, columns, length of a row and products call for (gemm_slim_impl.h), on 256 CUs."""
    import ruzinex_cases as Z

    class Zeros:  # (nothing is computed)
        standard_normal = staticmethod(lambda shape: np.zeros(shape, np.float32))
    np.random.default_rng = lambda seed: Zeros

    def forms(s, rows, want=1):
        stub.forget()
        step(s, 'a', rows, want)
        found = [re.search(r'slim_(group)_kernelILi(\d)|slim_kernel.*ShapeILi(\d+)ELi(\d)ELi(\d)ELi(\d)', k) for k in stub.kernels()]
        return [m[2] if m[1] else tuple(map(int, m.groups()[2:])) for m in found if m]

    for n, k, shapes in ((16384, 64, ((16, 2, 1, 2), (16, 2, 1, 4), (16, 2, 1, 8))), (16384, 512, ((16, 2, 1, 2), (16, 2, 1, 4), (16, 2, 1, 8))),
                         (16384, 2040, ((16, 2, 1, 2), (16, 2, 2, 4), (16, 2, 1, 8))), (16384, 2048, ((8, 4, 1, 4), (16, 2, 2, 4), (16, 2, 1, 8))),
                         (16384, 2056, ((16, 4, 2, 2), (16, 4, 2, 4), (16, 2, 1, 8))), (16385, 2056, ((16, 4, 2, 2), (16, 4, 2, 4), (16, 2, 2, 8))),
                         (16368, 64, ((16, 2, 2, 2), (16, 2, 2, 4), (16, 2, 1, 8))), (12288, 64, ((16, 2, 2, 2), (16, 2, 2, 4), (16, 2, 2, 8))),
                         (5504, 1536, ((16, 2, 2, 2), (16, 2, 2, 4), (16, 2, 2, 8))), (4096, 256, ((16, 2, 2, 2), (16, 4, 2, 4), (16, 4, 2, 8))),
                         (4096, 264, ((16, 8, 2, 2), (16, 4, 2, 4), (16, 4, 2, 8))), (2048, 264, ((8, 4, 2, 4), (16, 4, 2, 4), (16, 4, 2, 8)))):
        s = engine(Z.make_config([Z.layer(heads=2, kv_heads=1, dim=32, vdim=32)], width=k, vocab=n), Z, max_tokens=256, max_sequences=1)
        for rows, shape in zip(((2, 8), (9, 16), (17, 31)), shapes):
            assert [forms(s, m, m)[-1] for m in rows] == [shape] * 2, (n, k, rows)
    # 32 experts that all tokens go to: gated columns, then the width's
    for ff, width, want in ((520, 1032, ('1', '1', '1', '1', '2', '2')), (520, 2056, ((16, 4, 2, 2), '1', '1', '1', '2', '2')),
                            (128, 512, ((16, 2, 2, 2), (16, 2, 1, 2), (16, 2, 2, 4), '1', (16, 2, 2, 8), '2'))):
        mlp = Z.moe(experts=32, top=32, ff=ff, shared=0)
        s = engine(Z.make_config([Z.layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=mlp)], width=width), Z, max_tokens=256, max_sequences=1)
        got = tuple(f for m in (8, 16, 31) for f in forms(s, m, 0)[-2:])
        assert got == want, (ff, width, got)


def lone_choices(stub):
    """A lone token's products choose for themselves up to 64 outputs and 8 choices; beyond, a launch orders the pairs."""
    import ruzinex_cases as Z
    for experts, top, lone in ((1, 1, True), (8, 8, True), (64, 8, True), (64, 9, False), (9, 9, False), (64, 64, False), (65, 2, False)):
        s = engine(Z.make_config([Z.layer(mlp=Z.moe(experts=experts, top=top, ff=24))]), Z, max_tokens=256, max_sequences=1)
        stub.forget()
        step(s, 'a', 1, 0)
        assert any('lone_up_kernel' in k for k in stub.kernels()) == lone, (experts, top)


def group_tiles(stub):
    """Tiles of grouped products by rounds of 256 workgroups: a few tiles beyond whole rounds are no round."""
    import ruzinex_cases as Z
    for experts, top, tokens, ff, want in ((32, 2, 1700, 1024, (128, 256)), (16, 2, 1021, 1408, (128, 256)), (16, 8, 700, 2048, (128, 256)),
                                           (32, 2, 2048, 1024, (256, 256)), (16, 2, 1200, 1408, (256, 256)), (32, 4, 1700, 1024, (256, 256))):
        mlp = Z.moe(experts=experts, top=top, ff=ff, shared=0)
        s = engine(Z.make_config([Z.layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=mlp)], width=64), Z, max_tokens=4096, max_sequences=1)
        stub.forget()
        step(s, 'a', tokens, 0)
        found = [re.search(r'gemm_glds_kernelILi\d+ELi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)', k) for k in stub.kernels()]
        shapes = [(32 * int(m[1]) * int(m[3]), 32 * int(m[2]) * int(m[4])) for m in found if m]
        assert shapes[-2] == want, (experts, top, tokens, ff, shapes)


def tall_tiles(stub):
    """Which of test_gpu_group_tiles.py's products with rows of 512 values and more take tiles of up to 288 x 192: (gated columns, the width's)."""
    import ruzinex_cases as Z
    for width in (512, 576):
        mlp = Z.moe(experts=8, top=8, ff=2944, shared=0)
        s = engine(Z.make_config([Z.layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=mlp)], width=width), Z, max_tokens=1024, max_sequences=1)
        for tokens, want in ((72, (True, True)), (97, (False, True)), (129, (True, False)), (288, (True, False)), (330, (True, False))):
            stub.forget()
            step(s, 'a', tokens, 0)
            found = [k for k in stub.kernels() if re.search(r'gemm_glds_kernelI|wide_kernelI', k)]
            assert tuple('4tall16gemm_glds_kernelILi4ELi9ELi6ELi1ELi1E' in k for k in found[-2:]) == want, (width, tokens, found[-2:])
        s.release('a')


def tall_ungated_tiles(stub):
    """Experts without a gate on tall tiles, whose results leave as they are: the sizes of test_gpu_group_tiles.py."""
    import sodudra_cases as S
    import test_gpu_group_tiles as G

    class Zeros:  # (nothing is computed)
        standard_normal = staticmethod(lambda shape: np.zeros(shape, np.float32))
    np.random.default_rng = lambda seed: Zeros
    s = engine(G.ungated_config(S), S, max_tokens=1024, max_sequences=1)
    for tokens in G.UNGATED_ROWS:
        stub.forget()
        step(s, 'a', tokens, 0)
        assert any('4tall16gemm_glds_kernelILi4ELi9ELi6ELi1ELi1ELi0E' in k for k in stub.kernels()), tokens


def expected_rows(stub):
    """Tiles of grouped products follow the rows that a group is expected to have: choices of identity experts are none; a little over two tiles of 128 x 256 rather than two of 256 x 256."""
    import rofozen_cases as M
    import ruzinex_cases as Z

    class Zeros:  # (nothing is computed)
        standard_normal = staticmethod(lambda shape: np.zeros(shape, np.float32))
        uniform = staticmethod(lambda lo, hi, size=None: np.full(size, lo, np.float32))
    np.random.default_rng = lambda seed: Zeros

    def forms(cases, layer, width, tokens):
        s = engine(cases.make_config([layer], width=width), cases, max_tokens=4096, max_sequences=1)
        stub.forget()
        step(s, 'a', tokens, 0)
        return tuple(k for k in stub.kernels() if re.search(r'gemm_glds_kernelI.*Lb1E|tall|wide_kernelI.*Lb1E', k))[-2:]

    mamba = dict(heads=2, vdim=8, state=16, groups=1)
    for tokens in (96, 160, 200):
        with_identity = forms(M, M.mamba_layer(**mamba, mlp=M.moe(experts=8, identity=8, top=8, count=1, keep=1, ff=576)), 512, tokens)
        half, all_ = (forms(M, M.mamba_layer(**mamba, mlp=M.moe(experts=8, identity=0, top=top, count=1, keep=1, ff=576)), 512, tokens) for top in (4, 8))
        assert with_identity == half, (tokens, with_identity, half)
        assert tokens != 160 or half != all_, (half, all_)
    layer = Z.layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=Z.moe(experts=32, top=4, ff=1408, shared=0))
    for tokens, want in ((1600, 'wide_kernelILi4'), (2304, 'gemm_glds_kernelILi4ELi2ELi4ELi2ELi2E'), (2560, 'gemm_glds_kernelILi4ELi2ELi4ELi2ELi2E')):
        assert want in forms(Z, layer, 2048, tokens)[-1], (tokens, forms(Z, layer, 2048, tokens))


def walks_of_portions(stub):
    """Chunked recurrences take the walk of eight chunks a turn where the longest entry fills its turns and there are no more workgroups than the CUs have room for; the sizes of
    test_gpu_chunked_recurrences.py."""
    import rofozen_cases as M
    import test_gpu_chunked_recurrences as G
    import tolenex_cases as H

    class Zeros:  # (nothing is computed)
        standard_normal = staticmethod(lambda shape: np.zeros(shape, np.float32))
        uniform = staticmethod(lambda lo, hi, size=None: np.full(size, lo, np.float32))
    np.random.default_rng = lambda seed: Zeros

    def eight(cases, layer, entries):
        s = engine(cases.make_config([layer]), cases, max_tokens=sum(entries) + 64 * len(entries), max_sequences=len(entries), max_batch_tokens=sum(entries))
        stub.forget()
        s.step([(i, [1] * n, []) for i, n in enumerate(entries)])
        walks = [k for k in stub.kernels() if 'chunk_walk_kernel' in k]
        assert len(walks) == 1
        return 'eight_chunk_walk_kernel' in walks[0]

    def hgrn2(heads, dim, vdim):
        return H, H.hgrn2_layer(heads=heads, dim=dim, vdim=vdim)

    def mamba2(heads, dim, vdim):
        return M, M.mamba_layer(heads=heads, vdim=vdim, state=dim, groups=2)

    # up to one workgroup a CU
    for kind in (hgrn2, mamba2):
        for rows, want in ((32, False), (112, False), (113, True), (128, True), (129, False), (208, False), (209, True), (256, True), (257, False), (304, False), (305, True), (384, True),
                           (385, False), (400, False), (401, True), (497, True), (1021, True)):
            assert eight(*kind(16, 128, 128), [rows]) == eight(*kind(16, 128, 128), [rows, 1]) == want, (kind, rows)
        for dim in (192, 256):
            assert not eight(*kind(2, dim, 16), [1024])
    # more of them
    for kind, rows, want in ((hgrn2, 1024, False), (mamba2, 1024, True), (mamba2, 384, True), (mamba2, 385, False), (mamba2, 368, False), (mamba2, 368 + 1, True), (mamba2, 256, False)):
        assert eight(*kind(16, 128, 128), [rows] * 3) == eight(*kind(16, 128, 128), [rows] + [1] * 3) == want, (kind, rows)
        assert not eight(*kind(16, 128, 128), [rows] * 5) and not eight(*kind(16, 128, 128), [rows] + [1] * 7)
    # 64 rows of state
    for kind, rows, want in ((hgrn2, 704, False), (hgrn2, 720, False), (hgrn2, 721, True), (hgrn2, 768, True), (hgrn2, 769, False), (mamba2, 368, False), (mamba2, 384, True), (mamba2, 721, True)):
        assert eight(*kind(16, 64, 64), [rows]) == want, (kind, rows)
        assert not eight(*kind(16, 64, 64), [rows] * 5)
    for dim, steps in G.EIGHT_CHUNKS.items():
        for kind in (hgrn2, mamba2):
            assert [eight(*kind(4, dim, 16), [n for _, n in step]) for step in steps] == [len(step) > 1 for step in steps], (dim, kind)
    assert eight(*hgrn2(2, 128, 16), [113, 20]) and eight(*mamba2(4, 128, 16), [113, 20])


def who_sums(stub):
    """The experts' rows of few tokens are summed by the norm behind them, very many of them by a launch of its own."""
    import narurax_cases as N
    import ruzinex_cases as Z

    class Zeros:  # (nothing is computed)
        standard_normal = staticmethod(lambda shape: np.zeros(shape, np.float32))
        integers = staticmethod(lambda *a, **k: np.zeros(k.get('size', a[-1] if a else 1), np.int64))
        uniform = staticmethod(lambda lo, hi, size=None: np.full(size, lo, np.float32))
    np.random.default_rng = lambda seed: Zeros
    for width, top, tokens, apart in ((2048, 64, 1, False), (2056, 64, 1, True), (2056, 64, 64, True), (2056, 64, 65, False), (4104, 32, 8, True), (4104, 31, 8, False)):
        for cases, layer in ((Z, Z.layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=Z.moe(experts=64, top=top, ff=8, shared=0))),
                             (N, N.attn_layer(heads=2, kv_heads=1, dim=32, mlp=N.moe(experts=64, top=top, ff=8)))):
            s = engine(cases.make_config([layer], width=width), cases, max_tokens=256, max_sequences=1)
            stub.forget()
            step(s, 'a', tokens)
            assert any('moe_combine' in k for k in stub.kernels()) == apart, (width, top, tokens, cases)


def lone_row_forms(stub):
    """One row through experts that an ordering launch has looked up (over 64 outputs): a row of W by one wave or several, in one portion or more, by its
    length and by how many there are (pick_row_shape of stack_gemm.hip)."""
    import ruzinex_cases as Z

    class Zeros:  # (nothing is computed)
        standard_normal = staticmethod(lambda shape: np.zeros(shape, np.float32))
    np.random.default_rng = lambda seed: Zeros
    for width, ff, want in ((2048, 8, (1, 4)), (2056, 8, (2, 3)), (3072, 8, (2, 3)), (3080, 8, (2, 4)), (2056, 64, (2, 3)), (2056, 72, (1, 6)), (2056, 128, (1, 6)),
                            (2056, 136, (1, 3))):
        cfg = Z.make_config([Z.layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=Z.moe(experts=65, top=32, ff=ff, shared=0))], width=width)
        s = engine(cfg, Z, max_tokens=256, max_sequences=1)
        stub.forget()
        step(s, 'a', 1, 0)
        found = [re.search(r'row_kernelILi(\d)ELi(\d)', k) for k in stub.kernels()]
        assert [tuple(map(int, m.groups())) for m in found if m][-1] == want, (width, ff)  # (the down products: row_short_kernel)
    for columns, k, short in ((10752, 256, False), (10753, 256, True), (10753, 264, False), (16384, 512, False), (16385, 512, True), (16385, 520, False)):
        s = engine(Z.make_config([Z.layer(heads=2, kv_heads=1, dim=32, vdim=32)], width=k, vocab=columns), Z, max_tokens=256, max_sequences=1)
        stub.forget()
        step(s, 'a', 1)
        assert any('row_short_kernel' in k for k in stub.kernels()) == short, (columns, k)


if __name__ == '__main__':
    globals()[sys.argv[2]](Stub(sys.argv[1]), *sys.argv[3:])
    print('ok')
else:
    def test_scratch_of_the_state_layers(stub):
        run(stub, 'scratch_of_the_state_layers')

    def test_a_step_fits_where_only_the_optional_scratch_does_not(stub):
        run(stub, 'scratch_that_leaves_room')

    def test_a_step_behind_one_that_found_no_memory(stub):
        run(stub, 'step_behind_one_that_found_no_memory')

    def test_pinned_rows(stub):
        run(stub, 'pinned_rows')

    def test_steps_on_streams_in_turn(stub):
        run(stub, 'streams_in_turn')

    def test_who_waits_for_a_steps_rows(stub):
        run(stub, 'who_waits')

    def test_rows_that_end_where_memory_does(stub):
        run(stub, 'rows_to_the_edge')

    def test_a_step_with_more_tiles_than_a_grid_dimension(stub):
        run(stub, 'huge_step')

    def test_more_wanted_rows_than_a_grid_dimension(stub):
        run(stub, 'many_small_rows')

    def test_tile_shapes_of_the_product_tests(stub):
        run(stub, 'tile_shapes')

    def test_norms_without_an_experts_sum_do_not_carry_its_code(stub):
        run(stub, 'norms_without_a_sum')

    def test_forms_of_products_of_few_rows(stub):
        run(stub, 'few_row_forms')

    def test_forms_of_a_lone_row_through_groups(stub):
        run(stub, 'lone_row_forms')

    def test_who_chooses_for_a_lone_token(stub):
        run(stub, 'lone_choices')

    def test_who_sums_the_experts_rows(stub):
        run(stub, 'who_sums')

    def test_tall_tiles_of_grouped_products(stub):
        run(stub, 'tall_tiles')

    def test_tall_tiles_of_ungated_experts(stub):
        run(stub, 'tall_ungated_tiles')

    def test_expected_rows_of_grouped_products(stub):
        run(stub, 'expected_rows')

    def test_walks_of_portions(stub):
        run(stub, 'walks_of_portions')

    def test_tiles_of_grouped_products(stub):
        run(stub, 'group_tiles')

    def test_convolution_of_single_rows(stub):
        run(stub, 'convolution_of_single_rows')

    def test_lone_norms(stub):
        run(stub, 'lone_norms')

    def test_shifts_and_starts(stub):
        run(stub, 'shifts_and_starts')

    def test_packed_prompts(stub):
        run(stub, 'packed_prompts')

    def test_two_int8_products(stub):
        run(stub, 'two_int8_products')

    def test_int8_products(stub):
        run(stub, 'int8_products')

    def test_cold_weights_of_measured_products(stub):
        run(stub, 'cold_weights')

    def test_low_rank_pairs(stub):
        run(stub, 'low_rank_pairs')

    def test_sizes_of_the_row_tile_tests(stub):
        run(stub, 'row_tiles')

    def test_sizes_of_the_wide_tile_tests(stub):
        run(stub, 'wide_tiles')
