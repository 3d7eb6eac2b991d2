"""What StackEngine.step hands to the native engine, and what it hands back: no GPU, the native side is a recorder."""
import ctypes

import numpy as np
import pytest

from tensorrt_llm.runtime import stack


class Recorder:
    """tllm_stack_step that keeps the batch it is given and fills the rows with their numbers."""

    def __init__(self, vocab):
        self.vocab = vocab

    def tllm_stack_step(self, handle, batch, logits, ids, stream):
        b = batch._obj

        def ints(p, n):
            return [] if not n else list((ctypes.c_int32 * n).from_address(p))
        names = [f[0] for f in stack.Batch._fields_]
        n, e, w, blocks = (getattr(b, k) for k in names[:4])
        self.got = [ints(getattr(b, k), c) for k, c in zip(names[4:], (n, e, e, e, e * blocks, w))]
        if logits:
            np.ctypeslib.as_array((ctypes.c_float * (w * self.vocab)).from_address(logits))[:] = np.arange(w * self.vocab)
        if ids:
            np.ctypeslib.as_array((ctypes.c_int32 * w).from_address(ids))[:] = np.arange(w)
        return 0

    def tllm_stack_destroy(self, handle):
        pass


@pytest.fixture
def engine(monkeypatch):
    lib = Recorder(7)
    monkeypatch.setattr(stack, 'load_library', lambda *a, **k: lib)
    e = object.__new__(stack.StackEngine)
    e._h, e.vocab, e.lib = 1, lib.vocab, lib
    yield e
    e._h = None


WANT = [[5, 6, 7, 8], [3, 1], [0, 9], [1, 0], [4, 2, 0, 11, 12, 13], [2, 3]]
FORMS = {'lists': list, 'int32': lambda v: np.array(v, np.int32), 'int64': lambda v: np.array(v, np.int64), 'columns': lambda v: np.array(v, np.int32)[:, None],
         'strided': lambda v: np.repeat(np.array(v, np.int64), 2)[::2], 'blocks': lambda v: np.array(v)[:, None, None], 'floats': lambda v: np.array(v, np.float32)}


@pytest.mark.parametrize('form', FORMS)
def test_vectors_of_every_form_reach_the_engine(engine, form):
    f = FORMS[form]
    vectors = [f(v) for v in WANT[:4]]
    for table in (np.array(WANT[4]).reshape(2, 3), np.array(WANT[4], np.int32).reshape(3, 2).T.copy(), [WANT[4][:3], WANT[4][3:]],
                  np.asfortranarray(np.array(WANT[4], np.int16).reshape(2, 3))):
        logits, ids = engine.step(*vectors, table, f(WANT[5]))
        want = WANT[:4] + [np.asarray(table).reshape(-1).tolist(), WANT[5]]
        assert engine.lib.got == want
        assert logits.shape == (2, 7) and logits.dtype == np.float32 and (logits == np.arange(14).reshape(2, 7)).all() and ids.tolist() == [0, 1]


def test_no_wanted_rows(engine):
    logits, ids = engine.step(*WANT[:4], [[1], [2]], [])
    assert logits is None and ids.shape == (0,) and engine.lib.got[5] == []


@pytest.mark.parametrize('bad', [2 ** 31, 7.9, np.int64(-2 ** 31 - 1), True])
def test_lists_that_are_no_whole_numbers_of_32_bits_reach_the_engine_as_numpy_casts_them(engine, bad):
    tokens = [5, bad, 7, 8]
    table = np.array(WANT[4], np.int32).reshape(2, 3)
    table.flags.writeable = False
    engine.step(tokens, *WANT[1:4], table, WANT[5])
    want = np.empty(4, np.int32)
    want[:] = np.asarray(tokens)
    assert engine.lib.got == [want.tolist()] + WANT[1:]


def test_a_table_off_its_alignment_is_copied(engine):
    room = np.zeros(4 * 6 + 1, np.uint8)
    table = room[1:].view(np.int32).reshape(2, 3)
    table[...] = np.reshape(WANT[4], (2, 3))
    assert not table.flags.aligned and table.flags.c_contiguous
    at, take = [], engine.lib.tllm_stack_step
    engine.lib.tllm_stack_step = lambda handle, batch, *a: at.append(batch._obj.block_table) or take(handle, batch, *a)
    engine.step(*WANT[:4], table, WANT[5])
    assert engine.lib.got == WANT and at[0] % 4 == 0
