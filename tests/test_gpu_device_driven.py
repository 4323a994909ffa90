"""The step driven from the device (qd_k_lean.hpp) at the edges of its tiles,
bucket layouts and rooms, bit for bit against the oracle, and against the
host-driven path (qd_tuning.eager_select) where the oracle would take long."""
import math

import numpy as np
import pytest

import quids_amd as q
from oracle import oracle as orc
from quids_amd.rules import qcgd
from quids_amd.rules import quantum_computer as qc
from quids_amd.state import HostState

from helpers import assert_states_identical, qcgd_initial, sparse_graph

pytestmark = pytest.mark.gpu


def _registers(n, equal=False):
    """n distinct registers of 4 bytes: the qubit that the gate acts on and a
    number of 20 bits; random or equal magnitudes."""
    rng = np.random.default_rng(n)
    v = rng.permutation(1 << 20)[:n].astype(np.uint32)
    obj = np.zeros((n, 8), np.uint8)
    for k in range(3):
        obj[:, 1 + k] = (v >> (8 * k)) & 0xFF
    obj[:, 0] = rng.integers(0, 2, n)  # the qubit the gate acts on
    mag = rng.normal(size=n) + 1j * rng.normal(size=n)
    if equal:
        mag = np.full(n, 1 + 0j)
    return HostState(obj.reshape(-1), np.arange(n + 1, dtype=np.uint64) * np.uint64(8), np.full(n, 4, np.uint32),
                     mag / np.linalg.norm(mag))


def _step(hs, rule, cap, **tuning):
    ctx = q.default_context()
    old = ctx.get_tuning()
    ctx.set_tuning(**tuning)
    try:
        a, b = q.it_t(), q.it_t()
        a.upload(hs)
        out = []
        for _ in range(2):  # a fresh output state, then one that has room
            st = q.simulate(a, rule, b, None, cap)
            out.append(b.download())
        assert_states_identical(out[0], out[1], "repeated")
        return out[1], st
    finally:
        ctx.set_tuning(**{k: old[k] for k in tuning})


# candidates 2n: around the generate's chunk (1024), the order's tile (4096),
# the bucket layouts (128 per bucket, one pass of 480 x 256, the sub-buckets)
@pytest.mark.parametrize("n", [1, 63, 64, 65, 511, 512, 513, 2047, 2048, 2049, 16384, 16385, 61440, 61441, 140000])
def test_hadamard_sizes(n):
    hs = _registers(n)
    for cap in (q.UINT64_MAX, 2 * n, max(1, n + n // 3), max(1, n)):
        g, st = _step(hs, qc.hadamard(0), cap)
        o, ost = orc.simulate(hs, qc.hadamard(0), cap)
        assert (st["num_candidates"], st["num_unique"]) == (2 * n, ost["num_unique"])
        assert_states_identical(g, o, f"n {n} cap {cap}")


# as many equal |m|^2 as the finishing block takes, one more, and many
@pytest.mark.parametrize("n", [100, 4096, 4097, 30000])
def test_equal_magnitudes(n):
    hs = _registers(n, equal=True)
    for cap in (n, n + n // 2):
        g, _ = _step(hs, qc.hadamard(0), cap)
        o, _ = orc.simulate(hs, qc.hadamard(0), cap)
        assert_states_identical(g, o, f"equal {n} cap {cap}")


# parents around the number up to which the host does not wait for the
# candidates' number, with few candidates, and more than it made room for
@pytest.mark.parametrize("parents", [40, 2047, 2048, 2049])
@pytest.mark.parametrize("nodes", [7, 11])
@pytest.mark.parametrize("rule", [qcgd.split_merge(0.8, 0.3), qcgd.erase_create(1.1, 0.5), qcgd.coin(0.9, 0.2)])
def test_qcgd_parents(parents, nodes, rule):
    hs = qcgd_initial(nodes, 42)
    for r in (qcgd.split_merge(0.7, 0.2), qcgd.erase_create(1.0, 0.4)) * 2:
        hs = orc.simulate(hs, r, parents)[0]
        hs = orc.apply_modifier(hs, qcgd.step)
    for cap in (max(hs.num_object, 1000), q.UINT64_MAX):
        if cap == q.UINT64_MAX and nodes == 11 and parents > 40:
            continue
        g, st = _step(hs, rule, cap)
        o, ost = orc.simulate(hs, rule, cap)
        assert (st["num_candidates"], st["num_unique"]) == (ost["num_candidates"], ost["num_unique"])
        assert_states_identical(g, o, f"{type(rule).__name__} {parents} cap {cap}")


# 0.7e6 to 2e7 candidates: one child per lane, by work items, and beyond what
# the device drives
@pytest.mark.parametrize("parents", [9000, 60000, 150000])
def test_large_steps_match_the_host_driven_path(parents):
    a, b = q.it_t(), q.it_t()
    a.upload(HostState.from_objects([qcgd.seeded_graph(12, 42)]))
    rules = [qcgd.split_merge(math.pi / 4, 0.1), qcgd.erase_create(math.pi / 3, math.pi / 5)]
    for k in range(5):
        if k % 2 == 0:
            q.simulate(a, qcgd.step)
        q.simulate(a, rules[k % 2], b, None, parents // 4 if k < 4 else parents)
        a, b = b, a
    hs = a.download()
    got = {}
    for eager in (0, 1):
        for i, r in enumerate(rules):
            got[eager, i], _ = _step(hs, r, parents, eager_select=eager)
    for i in range(2):
        assert_states_identical(got[0, i], got[1, i], f"{parents} rule {i}")


# survivors' bytes: graphs around the lane segments' widths (16, 32, 64 nodes;
# beyond, the whole step runs on the generic kernels), children beyond the
# lists of 64 nodes, at every alignment
@pytest.mark.parametrize("align", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("nodes", [(1, 2), (15, 16), (16, 17), (31, 32, 33), (60, 63, 64), (64, 65)])
def test_populate_widths(nodes, align):
    old = q.align_byte_length
    q.align_byte_length = align
    try:
        objs = []
        for n in nodes:
            objs.append(sparse_graph(n, tuple(range(0, n, max(n // 5, 1))), ()))
            objs.append(sparse_graph(n, (n // 2,), (n // 3,) if n > 3 else ()))
        hs = HostState.from_objects(objs, align=align)
        for k, r in enumerate((qcgd.split_merge(0.8, 0.3), qcgd.coin(0.9, 0.2)) * 3):
            a, b = q.it_t(), q.it_t()
            a.upload(hs)
            q.simulate(a, r, b, None, 3000)
            ref, _ = orc.simulate(hs, r, 3000, align=align)
            assert_states_identical(b.download(), ref, f"{nodes} align {align} step {k}")
            hs = orc.apply_modifier(ref, qcgd.step)
    finally:
        q.align_byte_length = old


@pytest.mark.parametrize("size", [1, 3, 8, 9, 17, 64, 200])
def test_populate_register_sizes(size):
    rng = np.random.default_rng(size)
    objs = {bytes(rng.integers(0, 2, size).astype(np.uint8)) for _ in range(300)}
    hs = HostState.from_objects(sorted(objs))
    for bit in {0, size // 2, size - 1}:
        g, _ = _step(hs, qc.hadamard(bit), q.UINT64_MAX)
        o, _ = orc.simulate(hs, qc.hadamard(bit))
        assert_states_identical(g, o, f"size {size} bit {bit}")


# hashes that hundreds of candidates share, beyond a sub-bucket's fixed
# capacity: the entries beyond it go through the overflow list; a list that
# is full makes the pass repeat with exact counts
@pytest.mark.parametrize("copies,exact", [(690, False), (1500, False), (9000, True)])
@pytest.mark.parametrize("eager", [0, 1])
def test_overflowing_sub_buckets(copies, exact, eager):
    grown = qcgd_initial(12, 42)
    for r in (qcgd.split_merge(0.7, 0.2), qcgd.erase_create(1.0, 0.4)) * 2:
        grown = orc.simulate(grown, r, 2500)[0]
        grown = orc.apply_modifier(grown, qcgd.step)
    rng = np.random.default_rng(copies)
    objs = grown.objects_list() + [qcgd.seeded_graph(7, 5)] * copies
    mags = np.concatenate([grown.magnitude, 0.02 * (rng.normal(size=copies) + 1j * rng.normal(size=copies))])
    hs = HostState.from_objects(objs, mags)
    rule = qcgd.erase_create(0.8, 0.3)
    o, ost = orc.simulate(hs, rule, 20000)
    assert ost["num_candidates"] > 170000
    g, st = _step(hs, rule, 20000, eager_select=eager)
    assert st["num_unique"] == ost["num_unique"]
    assert bool(st["reserved"] & 1) == exact or st["reserved"] & 8
    assert_states_identical(g, o, f"copies {copies}")


def test_populate_long_names():
    """Children whose names grow from 36 sub_nodes past the lists' 384."""
    hs = qcgd_initial(16, 42)
    names = []
    for k in range(80):
        rule = qcgd.split_merge(1.56, 0.3) if k % 2 == 0 else qcgd.coin(0.3, 0.4)
        ref = orc.simulate(hs, rule, 12)[0]
        names.append(int(max(ref.object_size)) // 16)
        if k % 2 == 0 and k % 4 == 0:
            g, _ = _step(hs, rule, 12)
            assert_states_identical(g, ref, f"step {k}, {names[-1]} names")
        hs = orc.apply_modifier(ref, qcgd.step)
    assert max(names) > 400
