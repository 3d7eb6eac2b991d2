"""The rows that a step hands back belong to whoever asked for them (runtime/stack.py): no GPU, the native side is the recorder of
test_stack_step_arguments."""
import gc
import threading

import numpy as np

from test_stack_step_arguments import WANT, engine  # noqa: F401  (a fixture)


def rows(e):
    return e.step(*WANT[:4], np.array(WANT[4]).reshape(2, 3), WANT[5])[0]


def test_rows_own_their_memory(engine):  # noqa: F811
    a = rows(engine)
    assert a.base is None and a.flags.owndata and a.flags.c_contiguous and a.flags.writeable and type(a) is np.ndarray
    a.resize((3, 7))
    assert (a[:2] == np.arange(14).reshape(2, 7)).all() and (a[2] == 0).all()


def test_rows_of_one_step_are_not_those_of_another(engine):  # noqa: F811
    a = rows(engine)
    a[:] = 7.0
    view, buffer = a[1][2:5], memoryview(a)
    del a
    gc.collect()
    b = [rows(engine) for _ in range(50)]
    for x in b:
        x[:] = 1.0
    assert (view == 7.0).all() and (np.asarray(buffer) == 7.0).all()
    assert len({x.ctypes.data for x in b}) == 50


def test_threads(engine):  # noqa: F811
    bad = []

    def work(i):
        for _ in range(300):
            a = rows(engine)
            a[:] = i
            if not (a == i).all():
                bad.append(i)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(8)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad
