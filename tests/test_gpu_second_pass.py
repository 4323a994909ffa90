"""The second radix pass over its range of sub-bucket counts: up to 2^10 (two
workgroups a CU), 2^11 (one), beyond (entries written directly), and several
workgroups to a bucket in the hash-range passes, all the same final state as
the default layout."""
import math

import pytest

import quids_amd as q
from quids_amd.rules import qcgd
from quids_amd.state import HostState

from helpers import assert_states_identical

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def parents():
    """21672 graphs of 12 nodes: 1025244 children."""
    cur = q.it_t()
    cur.upload(HostState.from_objects([qcgd.seeded_graph(12, 4)]))
    rules = [qcgd.erase_create(math.pi / 3, math.pi / 5), qcgd.split_merge(math.pi / 4, 0.1)]
    for k in range(4):
        if k % 2 == 0:
            q.simulate(cur, qcgd.step)
        if k == 3:
            break
        nxt = q.it_t()
        q.simulate(cur, rules[k % 2], nxt)
        cur.close()
        cur = nxt
    yield cur, rules[1]
    cur.close()


def _final(parents, **tuning):
    ctx = q.default_context()
    old = ctx.get_tuning()
    cur, rule = parents
    ctx.set_tuning(**tuning)
    try:
        out = q.it_t()
        q.simulate(cur, rule, out, None, 20000)
        return out.download()
    finally:
        ctx.set_tuning(**{k: old[k] for k in tuning})


@pytest.mark.parametrize("first_pass_bits", [8, 4, 3, 2])
def test_sub_bucket_counts(parents, first_pass_bits):
    got = _final(parents, dedup_bucket_target=64, first_pass_bits=first_pass_bits)
    assert_states_identical(got, _final(parents), f"2^{first_pass_bits} buckets first")


@pytest.mark.parametrize("chunk_log2", [17, 19])
def test_range_groups(parents, chunk_log2):
    got = _final(parents, dedup_bucket_target=64, chunk_log2=chunk_log2)
    assert_states_identical(got, _final(parents), f"passes of 2^{chunk_log2}")
