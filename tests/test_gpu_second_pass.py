"""The partition and dedup over their ranges.  The second radix pass over its range of sub-bucket counts: up to 2^10 (two
workgroups a CU), 2^11 (one), beyond (entries written directly), and several
workgroups to a bucket in the hash-range passes, all the same final state as
the default layout."""
import math

import numpy as np
import pytest

import quids_amd as q
from oracle import oracle as orc
from quids_amd.rules import qcgd
from quids_amd.rules import quantum_computer as qc
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


# passes of several groups, whose pool is trimmed (a few of a group's uniques
# are above its bound)
@pytest.mark.parametrize("cap,chunk_log2", [(150000, 22), (300000, 24)])
def test_range_pool(parents, cap, chunk_log2):
    ctx = q.default_context()
    old = ctx.get_tuning()
    a, rule = q.it_t(), qcgd.erase_create(0.9, 0.4)
    q.simulate(parents[0], parents[1], a, None, cap)
    q.simulate(a, qcgd.step)
    out = {}
    try:
        for log2 in (0, chunk_log2):
            ctx.set_tuning(chunk_log2=log2)
            b = q.it_t()
            st = q.simulate(a, rule, b, None, cap)
            out[log2] = b.download()
            b.close()
            if log2:
                assert st["reserved"] & 4 and st["num_candidates"] > 2 << log2
    finally:
        ctx.set_tuning(chunk_log2=old["chunk_log2"])
        a.close()
    assert_states_identical(out[chunk_log2], out[0], f"cap {cap}")


# groups beyond the registers' eight members, in the LDS table of each size:
# ranked by one wavefront (up to 64 entries), by all threads (up to half of
# them), sorted beyond
@pytest.mark.parametrize("dedup_cap", [256, 512, 1024, 2048])
@pytest.mark.parametrize("copies", [9, 31, 32, 33, 63, 64, 65, 127, 128, 129, 240])
def test_groups_of_equal_hashes(copies, dedup_cap):
    rng = np.random.default_rng(copies)
    n = 4 * copies
    reg = np.zeros((n, 8), np.uint8)
    # a few registers share each hash: `copies` of one, and groups of 1 to 12
    kinds = np.concatenate([np.zeros(copies), 1 + rng.integers(0, n // 4, n - copies)]).astype(np.uint32)
    kinds = rng.permutation(kinds)
    reg[:, 1], reg[:, 2] = kinds & 0xFF, kinds >> 8
    reg[:, 0] = rng.integers(0, 2, n)
    mag = rng.normal(size=n) + 1j * rng.normal(size=n)
    hs = HostState(reg.reshape(-1), np.arange(n + 1, dtype=np.uint64) * np.uint64(8), np.full(n, 4, np.uint32),
                   mag / np.linalg.norm(mag))
    ctx = q.default_context()
    old = ctx.get_tuning()
    ctx.set_tuning(dedup_bucket_target=min(dedup_cap // 2, 512), dedup_cap=dedup_cap)
    try:
        a, b = q.it_t(), q.it_t()
        a.upload(hs)
        st = q.simulate(a, qc.hadamard(0), b)
        ref, ost = orc.simulate(hs, qc.hadamard(0))
        assert st["num_unique"] == ost["num_unique"]
        assert_states_identical(b.download(), ref, f"{copies} copies, table of {dedup_cap}")
    finally:
        ctx.set_tuning(dedup_bucket_target=old["dedup_bucket_target"], dedup_cap=old["dedup_cap"])


def test_small_steps_after_hash_range_passes(parents):
    """A hash-range step leaves its buffers with the context; the steps after
    it, among them one whose select the device hands back (more equal keys
    than one block takes), are the same as without them."""
    ctx = q.default_context()
    old = ctx.get_tuning()

    def chain():
        cur = q.it_t()
        cur.upload(HostState.from_objects([qcgd.seeded_graph(10, 42)]))
        for k in range(4):
            if k % 2 == 0:
                q.simulate(cur, qcgd.step)
            nxt = q.it_t()
            q.simulate(cur, [qcgd.split_merge(math.pi / 4, 0.0), qcgd.erase_create(math.pi / 3, math.pi / 5)][k % 2],
                       nxt, None, 1 << 18)
            cur.close()
            cur = nxt
        out = cur.download()
        cur.close()
        return out

    ref = chain()
    a = q.it_t()
    q.simulate(parents[0], parents[1], a, None, 150000)
    ctx.set_tuning(chunk_log2=22)
    try:
        b = q.it_t()
        st = q.simulate(a, qcgd.erase_create(0.9, 0.4), b, None, 150000)
        assert st["reserved"] & 4
        for s in (a, b):
            s.close()
    finally:
        ctx.set_tuning(chunk_log2=old["chunk_log2"])
    for k in range(2):
        assert_states_identical(chain(), ref, f"after a hash-range step, {k}")
