"""The memory behind a step's rows (runtime/stack.py): no GPU, no engine."""
import gc
import threading

import numpy as np

from tensorrt_llm.runtime.stack import _RowPool


def test_rows_are_handed_out_again_only_when_nobody_looks_at_them():
    pool = _RowPool()
    a, at = pool.rows(3, 50)
    assert a.shape == (3, 50) and a.dtype == np.float32 and a.ctypes.data == at and a.flags.c_contiguous and a.flags.writeable
    a[:] = 7.0
    view, buffer = a[1][10:20], memoryview(a)
    del a
    gc.collect()
    b, at_b = pool.rows(3, 50)
    assert at_b != at
    b[:] = 1.0
    assert (view == 7.0).all() and (np.asarray(buffer) == 7.0).all()
    del view
    assert pool.rows(3, 50)[1] not in (at, at_b)
    del buffer
    gc.collect()
    assert pool.rows(3, 50)[1] == at
    assert pool.rows(2, 50)[1] != at


def test_what_waits_is_bounded_and_other_sizes_give_way():
    pool = _RowPool()
    for n in (1, 2, 3):
        held = [pool.rows(n, 1 << 18)[0] for _ in range(40)]
        del held
        gc.collect()
        assert sum(k * len(v) for k, v in pool._idle.items()) <= pool.LIMIT
        assert pool._idle[n << 20]
    held = pool.rows(64, 1 << 18)[0]
    held[:] = 0.0
    del held
    assert sum(k * len(v) for k, v in pool._idle.items()) <= pool.LIMIT


def test_rows_outlive_their_pool():
    pool = _RowPool()
    a, _ = pool.rows(2, 30)
    a[:] = 5.0
    del pool
    gc.collect()
    assert (a == 5.0).all()


def test_threads():
    pool, bad = _RowPool(), []

    def work(i):
        for k in range(300):
            a, _ = pool.rows(1 + k % 3, 64)
            a[:] = i
            if not (a == i).all():
                bad.append(i)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(8)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad
