"""State buffers kept between uses (StatePool): results do not depend on where
a state's memory comes from, closing states from another thread is safe, the
pool is bounded and given back."""
import math
import threading

import numpy as np
import pytest
import torch

import quids_amd as q
from quids_amd.rules import qcgd
from quids_amd.state import HostState

from helpers import assert_states_identical

pytestmark = pytest.mark.gpu


def _chain(cap, n=5, keep=None):
    """The final state of n truncated steps, each into a state of its own."""
    cur = q.it_t()
    cur.upload(HostState.from_objects([qcgd.seeded_graph(9, 4)]))
    rules = [qcgd.split_merge(math.pi / 4, 0.1), qcgd.erase_create(math.pi / 3, math.pi / 5)]
    for k in range(2 * n):
        if k % 2 == 0:
            q.simulate(cur, qcgd.step)
        nxt = q.it_t()
        q.simulate(cur, rules[k % 2], nxt, None, cap)
        (keep.append if keep is not None else q.it_t.close)(cur)
        cur = nxt
    out = cur.download()
    cur.close()
    return out


def test_reused_buffers_give_the_same_states():
    ctx = q.default_context()
    ctx.trim()
    ref = _chain(30000)
    for cap in (30000, 500, 30000, 60000, 30000):
        got = _chain(cap)
        if cap == 30000:
            assert_states_identical(got, ref, "reused")
    # closed by another thread while this one goes on
    kept = []
    _chain(30000, keep=kept)
    t = threading.Thread(target=lambda: [s.close() for s in kept])
    t.start()
    got = _chain(30000)
    t.join()
    assert_states_identical(got, ref, "beside a closing thread")


def test_pool_is_bounded_and_given_back():
    ctx = q.default_context()
    obj = np.zeros(600 << 20, np.uint8)  # one object of 600 MB: pages that are never read cost nothing here
    ctx.trim()
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    states = []
    for _ in range(12):
        s = q.it_t()
        s.upload(HostState(obj, np.array([0, obj.size], np.uint64), np.array([16], np.uint32), np.ones(1, complex)))
        states.append(s)
    held = before - torch.cuda.mem_get_info()[0]
    assert held > 12 * obj.size
    for s in states:
        s.close()
    assert before - torch.cuda.mem_get_info()[0] <= (4 << 30) + (64 << 20)
    ctx.trim()
    assert before - torch.cuda.mem_get_info()[0] <= 64 << 20
