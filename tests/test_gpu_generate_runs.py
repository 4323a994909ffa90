"""Generate fused with the first radix pass (k_generate_scatter): chunks whose
parents' tables fit the LDS area and chunks whose do not, parents of one work
item and of many, at the edges of its chunks, with one to 2^9 buckets; bit for
bit against the oracle."""
import numpy as np
import pytest

import quids_amd as q
from oracle import oracle as orc
from quids_amd.rules import qcgd
from quids_amd.state import HostState

from helpers import assert_states_identical, sparse_graph

pytestmark = pytest.mark.gpu


def _parents(nodes, count):
    rng = np.random.default_rng(count)
    objs = {}
    while len(objs) < count:
        n = nodes[len(objs) % len(nodes)]
        ops = [tuple(sorted(rng.choice(m, size=min(m, int(rng.integers(1, 5))), replace=False).tolist()))
               for m in (n, n - 1)]
        objs[(n, *ops)] = sparse_graph(n, *ops)
    rng.shuffle(order := list(objs))
    return HostState.from_objects([objs[k] for k in order])


@pytest.mark.parametrize("first_pass_bits", [1, 8, 9])
@pytest.mark.parametrize("nodes,count", [((5,), 1), ((12,), 255), ((12,), 256), ((12, 13), 700), ((40,), 300),
                                         ((64,), 257), ((8, 64), 600)])
def test_chunks_of_parents(nodes, count, first_pass_bits):
    hs = _parents(nodes, count)
    ctx = q.default_context()
    old = ctx.get_tuning()
    # (small buckets and a first pass of its own: the host-driven path)
    ctx.set_tuning(dedup_bucket_target=64, first_pass_bits=first_pass_bits)
    try:
        rules = [qcgd.split_merge(0.8, 0.3)]
        if max(nodes) < 13:  # (a decision per empty node)
            rules.append(qcgd.erase_create(1.1, 0.5))
        for rule in rules:
            a, b = q.it_t(), q.it_t()
            a.upload(hs)
            st = q.simulate(a, rule, b, None, 5000)
            ref, ost = orc.simulate(hs, rule, 5000)
            assert st["num_candidates"] == ost["num_candidates"]
            assert_states_identical(b.download(), ref, f"{nodes} {count} {first_pass_bits}")
    finally:
        ctx.set_tuning(dedup_bucket_target=old["dedup_bucket_target"], first_pass_bits=old["first_pass_bits"])
