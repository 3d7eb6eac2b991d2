"""What a request starts from, brought over in one launch, and a step graph that outlives its request (session.cpp): requests one behind the other on one session and on another stream,
prompts of other lengths, ids that do not fill 16 bytes, another end token from request to request, requests that are not waited for."""
import numpy as np
import pytest
import torch

from test_gpu_ragged_prompts import NEW, sessions

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('batch,prompt', [(1, 5), (3, 9), (4, 16)])
def test_requests_do_not_depend_on_the_one_before(batch, prompt):
    many, session = sessions('fp16', 0)
    s, new = session(batch, prompt), NEW
    rng = np.random.default_rng(batch)
    requests = [(many[:batch, 17 * i:17 * i + prompt].copy(), rng.integers(1, prompt + 1, batch).astype(np.int32)) for i in range(4)]
    alone = []
    for ids, lens in requests:
        one = session(batch, prompt)
        alone.append(one.generate(ids, lens, new))
        one.close()
    for _ in range(2):
        for (ids, lens), want in zip(requests, alone):
            np.testing.assert_array_equal(s.generate(ids, lens, new), want)
    # another end token: the tokens behind it are that token, and it is no longer one in the next request
    ids, lens = requests[0]
    end = int(alone[0][0, prompt])
    cut = s.generate(ids, lens, new, end_id=end)
    assert (cut[0, prompt:] == end).all()
    np.testing.assert_array_equal(s.generate(ids, lens, new), alone[0])
    # a prompt phase that nobody waited for ahead of the next request, and requests on another stream
    s.context(*requests[1])
    np.testing.assert_array_equal(s.generate(ids, lens, new), alone[0])
    other = torch.cuda.Stream()
    s.context(*requests[2], stream=other.cuda_stream)
    np.testing.assert_array_equal(s.generate(*requests[3], new, stream=other.cuda_stream), alone[3])
    other.synchronize()
    np.testing.assert_array_equal(s.generate(ids, lens, new), alone[0])
    s.close()


@pytest.mark.parametrize('mode', ['fp16', 'sq_static_pc'])
def test_beam_requests_do_not_depend_on_the_one_before(mode):
    """The second request's steps are all replayed: its ids, its logits and how many rows of them there are, are the first one's."""
    many, session = sessions(mode, 0)
    s = session(2, 9)
    s.setup(2, 9, NEW, beam_width=3)
    ids, lens = many[:2, :9].copy(), np.array([9, 4], np.int32)
    got = []
    for prompt in (ids, many[2:4, :9].copy(), ids, ids):
        out = s.generate(prompt, lens, NEW)
        got.append((out, s.logits()))
        assert got[-1][1].shape[0] == 6
    for out, logits in got[2:]:
        np.testing.assert_array_equal(out, got[0][0])
        np.testing.assert_array_equal(logits, got[0][1])
    s.close()
