"""Host side of a LLaMA session's requests (session.cpp) over the stand-in for the HIP runtime (hip_stub.cpp), without a GPU: nothing is computed, but every allocation, launch, wait and
captured step is the real code's.  Each scenario runs in a process of its own, with the stand-in loaded ahead of the library."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

from test_stack_host_runtime import Stub, stub  # noqa: F401 (fixture)

S, NEW = 16, 6


def run(stub, scenario):  # noqa: F811
    r = subprocess.run([sys.executable, os.path.abspath(__file__), stub, scenario], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


# ------------------------------------------------------------------------------------------------------------ in the child process
def session(mode='fp16', batch=1, beam=1):
    import test_gpu_session as G
    from oracle import quant_oracle as QO
    from tensorrt_llm.runtime.native import NativeSession
    cfg, w = G.synth_model(7)
    ids = np.full((1, 8), 5, np.int32)
    m = QO.quantise_model(cfg, w, mode, 0, calib_ids=ids, calib_lens=np.array([8], np.int32))
    s = NativeSession(dict(cfg, quant_mode=m['quant_mode']))
    for k, v in m['engine_tensors'].items():
        s.set_tensor(k, v)
    s.finalize()
    s.setup(batch, S, NEW, beam_width=beam)
    return s


def request(s, **kw):
    return s.generate(np.full((s.batch, S), 3, np.int32), np.full(s.batch, S, np.int32), NEW, **kw)


def rows_of_logits(stub):  # noqa: F811
    """The logits behind a request are its last step's, whether its steps were launched or replayed; behind a prompt they are the prompts'."""
    for batch, beam in ((2, 3), (2, 1)):
        s = session(batch=batch, beam=beam)
        for stream in (0, 0, 64, 64):
            request(s, stream=stream)
            assert s.logits(stream=stream).shape[0] == batch * beam, (batch, beam, stream)
        for graph in (False, True, True):
            s.context(np.full((batch, S), 3, np.int32), np.full(batch, S, np.int32))
            s.step(0, use_graph=graph)
            assert s.logits().shape[0] == batch, (batch, beam, graph)
            s.step(2, use_graph=graph)
            assert s.logits().shape[0] == batch * beam, (batch, beam, graph)
        s.close()


def set_up_without_memory(stub):  # noqa: F811
    """A set-up that fails for want of memory, on the device or pinned, gives back what it made, and requests behind it are told to set up first."""
    s = session()
    request(s)
    s.setup(1, S, NEW)
    pinned = stub.pinned_bytes()
    assert pinned > 0
    weights = stub.live()  # (an upper bound: with the set-up)
    for what, size in (('budget', 0), ('budget', weights // 2), ('budget', weights - 4096), ('pinned_budget', pinned - 1)):
        getattr(stub, what)(size)
        with pytest.raises(RuntimeError, match='hipMalloc|hipHostMalloc'):
            s.setup(1, S, NEW)
        getattr(stub, what)(2 ** 64 - 1)
        assert stub.pinned_bytes() == 0 and stub.live() < weights, what
        s.batch, s.max_in, s.max_new = 1, S, NEW
        for call in (lambda: request(s), lambda: s.context(np.full((1, S), 3, np.int32), np.full(1, S, np.int32)), lambda: s.step(1)):
            with pytest.raises(RuntimeError, match='setup'):
                call()
        s.setup(1, S, NEW)
        request(s)
        assert stub.live() == weights and stub.pinned_bytes() == pinned, what
    s.close()
    assert stub.pinned_bytes() == 0


def knobs_between_requests(stub):  # noqa: F811
    """A request's steps are launched as the knobs of the decode products and its end token say at the time, and recorded anew only where one of them has changed."""
    from tensorrt_llm.plugin import capi
    lib = capi.load_library()
    s = session('sq_static_pc', batch=6)

    def kernels(**kw):
        stub.forget()
        request(s, **kw)
        return stub.kernels()

    def by_mfma(names):
        return sum('gemv_mfma' in n for n in names)

    first = kernels()
    assert by_mfma(first) > 0 and kernels() == first
    graphs = stub.graphs()
    assert kernels() == first and stub.graphs() == graphs
    lib.tllm_gemv_set_mfma_rows(0)
    by_rows = kernels()
    assert by_mfma(by_rows) == 0 and stub.graphs() == graphs + 1
    assert kernels() == by_rows and stub.graphs() == graphs + 1
    lib.tllm_gemv_set_blocks_per_cu(1)  # (the same kernels, by fewer workgroups)
    assert kernels() == by_rows and stub.graphs() == graphs + 2
    lib.tllm_gemv_set_blocks_per_cu(0)
    lib.tllm_gemv_set_mfma_rows(-1)
    assert kernels() == first and stub.graphs() == graphs + 3
    for end_id, new in ((400, 1), (400, 0), (-1, 1)):
        graphs = stub.graphs()
        assert kernels(end_id=end_id) == first and stub.graphs() == graphs + new, end_id
    # a step of the caller's own is replayed under the same rule
    for rows, mfma in ((0, False), (0, False), (5, True)):
        lib.tllm_gemv_set_mfma_rows(rows)
        s.context(np.full((6, S), 3, np.int32), np.full(6, S, np.int32))
        stub.forget()
        s.step(1, use_graph=True)
        assert (by_mfma(stub.kernels()) > 0) == mfma, rows
    s.close()


def prompts_on_streams_in_turn(stub):  # noqa: F811
    """A prompt waits until the one before it has been read from pinned memory, on whichever stream, and for nothing else on the device."""
    s = session()
    for stream in (0, 64, 64, 128, 0):
        before = stub.device_syncs(), stub.stream_syncs(), stub.event_syncs()
        s.context(np.full((1, S), 3, np.int32), np.full(1, S, np.int32), stream=stream)
        assert (stub.device_syncs(), stub.stream_syncs(), stub.event_syncs()) == (before[0], before[1], before[2] + 1), stream
    # a whole request waits for its tokens, and for its stream where it fails: nothing is left to be waited for
    records, before = stub.event_records(), stub.device_syncs()
    for stream in (64, 0):
        request(s, stream=stream)
    assert (stub.event_records(), stub.device_syncs()) == (records, before)
    streams = stub.stream_syncs()
    stub.fail_launches(1)
    with pytest.raises(RuntimeError, match='launch failed'):
        request(s)
    stub.fail_launches(0)
    assert (stub.event_records(), stub.device_syncs(), stub.stream_syncs()) == (records, before, streams + 1)
    s.context(np.full((1, S), 3, np.int32), np.full(1, S, np.int32))
    assert stub.event_records() == records + 1
    device, events = stub.device_syncs(), stub.event_syncs()
    s.close()
    assert stub.device_syncs() == device and stub.event_syncs() == events + 1  # (ahead of giving the memory back)


if __name__ == '__main__':
    sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
    globals()[sys.argv[2]](Stub(sys.argv[1]))
    print('ok')
else:
    def test_rows_of_logits(stub):  # noqa: F811
        run(stub, 'rows_of_logits')

    def test_set_up_without_memory(stub):  # noqa: F811
        run(stub, 'set_up_without_memory')

    def test_knobs_between_requests(stub):  # noqa: F811
        run(stub, 'knobs_between_requests')

    def test_prompts_on_streams_in_turn(stub):  # noqa: F811
        run(stub, 'prompts_on_streams_in_turn')
