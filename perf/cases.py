"""The workloads whose speed is followed: what a user of quids_amd has it do,
through its public entry points, from a few objects to steps beyond one
pass.

Kinds of case (a case is a dict of plain values):

* ``loop``: a driver loop from one graph, per iteration split_merge,
  erase_create, an observable of the state and the step modifier, as the
  reference's command line runs it (src/rules/qcgd.hpp:1168-1176).  Small
  states: launches and read-backs count.
* ``circuit``: a quantum_computer circuit, a Hadamard gate per qubit with
  CNOT, X, Y and Z gates between them; the state doubles with every gate.
* ``step``: one simulate() call on a state that earlier iterations grew and
  truncated, the call that a long QCGD run consists of.  With ``chunk_log2``
  the context takes at most 2^chunk_log2 candidates a pass, so that the step
  runs in hash-range passes, as a step beyond device memory does.
* ``walk``: one coin step (the quantum walk's) of a superposition of few
  particles on a wide ring.
* ``batch``: one iteration of many independent instances in two batched
  calls.
* ``gradient``: value and gradient of an expectation with respect to the
  rules' angles, with checkpoints.

A case's ``graph`` number places the particles, the seed sets the angles
and the magnitudes: inputs of every seed are other inputs of the same size.
"""
import ctypes
import math
import random

import numpy as np
import torch

import quids_amd as q
from quids_amd import adjoint as adj
from quids_amd import batch as qb
from quids_amd._abi import check, lib
from quids_amd.rules import qcgd
from quids_amd.rules import quantum_computer as qc
from quids_amd.state import HostState

UNLIMITED = q.UINT64_MAX


def listed():
    return [
        # the smallest program: two untruncated iterations of six nodes, some
        # thousands of candidates at most (the smoke size, and the command
        # line's examples)
        dict(name="loop_n6", kind="loop", nodes=6, iterations=2, cap=0, graph=4),
        # a small truncated run: what an interactive study of a few nodes does
        dict(name="loop_n9", kind="loop", nodes=9, iterations=4, cap=1000, graph=2),
        # a 16-qubit circuit (the tests' register)
        dict(name="circuit_q16", kind="circuit", qubits=16, gates=20, graph=3),
        # the walk of six particles on a ring of 40 nodes
        dict(name="walk_n40", kind="walk", nodes=40, particles=6, parents=10007, graph=4),
        # ordinary steps of 12 nodes, the tests' and the tuning's workload
        dict(name="split_n12", kind="step", rule="split_merge", nodes=12, parents=20000, cap=20000,
             probabilistic=False, chunk_log2=0, graph=3),
        dict(name="create_n12", kind="step", rule="erase_create", nodes=12, parents=50000, cap=50000,
             probabilistic=False, chunk_log2=0, graph=4),
        # large steps of 12 nodes in one pass, 1e8 to 2e8 candidates each
        dict(name="split_n12_large", kind="step", rule="split_merge", nodes=12, parents=1 << 21, cap=1 << 21,
             probabilistic=False, chunk_log2=0, graph=3),
        dict(name="create_n12_large", kind="step", rule="erase_create", nodes=12, parents=1 << 20, cap=1 << 20,
             probabilistic=False, chunk_log2=0, graph=3),
        # steps of 16 nodes in some 20 hash-range passes: the benchmark's
        # workload (bench.py) at a state size that is quick to make
        dict(name="range_split_n16", kind="step", rule="split_merge", nodes=16, parents=1 << 21, cap=1 << 21,
             probabilistic=False, chunk_log2=25, graph=3),
        dict(name="range_create_n16", kind="step", rule="erase_create", nodes=16, parents=1 << 20, cap=1 << 20,
             probabilistic=False, chunk_log2=26, graph=3),
        # 256 instances of 6 to 16 nodes advanced together
        dict(name="batch_256", kind="batch", instances=256, lo=6, hi=16, cap=1024, graph=7),
        # the gradient workload (bench.py): 10 nodes, 6 iterations
        dict(name="gradient_n10", kind="gradient", nodes=10, iterations=6, cap=1 << 16, checkpoint=2, graph=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["loop", "loop", "circuit", "walk", "step", "step", "step", "range", "batch", "gradient"])
    graph = rng.randrange(1 << 20)
    if kind == "loop":
        cap = rng.choice([0, _log_int(rng, 20, 20000), _log_int(rng, 20, 20000)])
        return dict(kind="loop", nodes=rng.randint(4, 12 if cap else 7), iterations=rng.randint(1, 4 if cap else 2),
                    cap=cap, graph=graph)
    if kind == "circuit":
        return dict(kind="circuit", qubits=rng.randint(3, 18), gates=rng.randint(3, 24), graph=graph)
    if kind == "walk":
        return dict(kind="walk", nodes=rng.randint(9, 60), particles=rng.randint(4, 7),
                    parents=_log_int(rng, 50, 20000), graph=graph)
    if kind == "batch":
        lo = rng.randint(5, 9)
        return dict(kind="batch", instances=rng.randint(2, 300), lo=lo, hi=lo + rng.randint(0, 6),
                    cap=_log_int(rng, 64, 1024), graph=graph)
    if kind == "gradient":
        return dict(kind="gradient", nodes=rng.randint(5, 10), iterations=rng.randint(1, 6),
                    cap=_log_int(rng, 1000, 1 << 16), checkpoint=rng.randint(1, 3), graph=graph)
    rule = rng.choice(["split_merge", "erase_create"])
    if kind == "range":
        nodes = rng.randint(12, 16)
        parents = _log_int(rng, 1 << 16, 1 << 20)
        return dict(kind="step", rule=rule, nodes=nodes, parents=parents, cap=parents + rng.randint(0, parents // 2),
                    probabilistic=False, chunk_log2=rng.randint(22, 26), graph=graph)
    nodes = rng.randint(6, 14)
    most = 2.5e8 / _children(rule, nodes)
    parents = _log_int(rng, 100, min(most, 1 << 21))
    return dict(kind="step", rule=rule, nodes=nodes, parents=parents, cap=parents + rng.randint(0, parents // 2),
                probabilistic=rng.random() < 0.25, chunk_log2=0, graph=graph)


# -- inputs ---------------------------------------------------------------
_contexts = {}


def _context(chunk_log2=0):
    """The program's context: the default one, or one whose steps take at
    most 2^chunk_log2 candidates a pass."""
    if not chunk_log2:
        return q.default_context()
    if chunk_log2 not in _contexts:
        _contexts.clear()  # one such context at a time: each holds its own scratch
        _contexts[chunk_log2] = q.Context(0)
        _contexts[chunk_log2].set_tuning(chunk_log2=chunk_log2)
    return _contexts[chunk_log2]


def _particles(nodes, rng):
    """Half of the left and half of the right places of a cycle, taken."""
    bits = [[1] * ((nodes + 1) // 2) + [0] * (nodes // 2) for _ in range(2)]
    for b in bits:
        rng.shuffle(b)
    return bits


def _graph(nodes, rng):
    return qcgd.with_particles(qcgd.make_graph(nodes), *_particles(nodes, rng))


def _angles(rng):
    """(theta, phi) of split_merge and of erase_create."""
    return [rng.uniform(0.2, 0.3) * math.pi, rng.uniform(0, 0.4) * math.pi,
            rng.uniform(0.25, 0.4) * math.pi, rng.uniform(0.1, 0.4) * math.pi]


def _rules(a):
    return [qcgd.split_merge(a[0], a[1]), qcgd.erase_create(a[2], a[3])]


def _grown(case, rules, ctx):
    """The state that `case`'s step acts on: three iterations truncated to a
    fraction of its parents, the last call before the step to all of them."""
    small = max(case["parents"] // (64 if case["nodes"] >= 14 else 4), 64)
    a, b = q.it_t(ctx=ctx), q.it_t(ctx=ctx)
    a.upload(HostState.from_objects([_graph(case["nodes"], random.Random(case["graph"]))]))
    calls = 6 if case["rule"] == "split_merge" else 7
    for k in range(calls):
        if k % 2 == 0:
            q.simulate(a, qcgd.step)
        q.simulate(a, rules[k % 2], b, None, small if k + 1 < calls else case["parents"])
        a, b = b, a
    if calls % 2 == 0:
        q.simulate(a, qcgd.step)
    b.close()
    return a


def _walk_state(case, seed):
    """Distinct placements of `particles` particles on the ring's 2n places:
    left and right masks, and random magnitudes of norm 1."""
    g = np.random.default_rng(case["graph"])
    n, N = case["nodes"], case["parents"]
    place = np.sort(np.argsort(g.random((N + N // 4 + 64, 2 * n)), axis=1)[:, :case["particles"]], axis=1)
    bit = np.where(place < n, np.uint64(1) << (place % n).astype(np.uint64), np.uint64(0))
    left = np.bitwise_or.reduce(bit, axis=1)
    bit = np.where(place >= n, np.uint64(1) << (place % n).astype(np.uint64), np.uint64(0))
    right = np.bitwise_or.reduce(bit, axis=1)
    _, first = np.unique(np.stack([left, right], 1).view("V16").reshape(-1), return_index=True)
    first = np.sort(first)[:N]
    g = np.random.default_rng(seed)
    mag = g.standard_normal(first.size) + 1j * g.standard_normal(first.size)
    return left[first], right[first], mag / np.sqrt(np.sum(np.abs(mag) ** 2))


def _walk_angles(seed):
    rng = random.Random(seed)
    return rng.uniform(0.2, 0.3) * math.pi, rng.uniform(0.1, 0.4) * math.pi, rng.uniform(0.1, 0.4) * math.pi


def _circuit(case, seed):
    """The register's first value, and [(gate, bits)]: Hadamards, each on a
    new qubit as long as there are any, and a random modifier after each."""
    rng = random.Random(case["graph"])
    bits = list(range(case["qubits"]))
    rng.shuffle(bits)
    gates = []
    for k in range(case["gates"]):
        gates.append(("h", bits[k] if k < len(bits) else rng.choice(bits)))
        gate = rng.choice(["cnot", "x", "y", "z"])
        gates.append((gate, *rng.sample(bits, 2)) if gate == "cnot" else (gate, rng.choice(bits)))
    rng = random.Random(seed)
    return [rng.randint(0, 1) for _ in bits], gates


def _outputs(state, it, most):
    """Gives the program tensors of its own for the object bytes, on the
    library's stream: their number is not the same for every input, so there
    is room for `most`."""
    stream = ctypes.c_void_p()
    check(lib().qd_ctx_stream(it.ctx.handle, ctypes.byref(stream)), "qd_ctx_stream")
    state["stream"] = torch.cuda.ExternalStream(stream.value)
    state["bytes"] = torch.zeros(most, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    return state


def prepare(case, seed):
    rng = random.Random(seed)
    kind = case["kind"]
    if kind == "loop":
        start = q.it_t()
        start.upload(HostState.from_objects([_graph(case["nodes"], random.Random(case["graph"]))]))
        state = dict(case=case, start=start, pair=(q.it_t(), q.it_t()), rules=_rules(_angles(rng)))
        return _outputs(state, start, (case["cap"] or 200000) * (200 * case["nodes"]))
    if kind == "circuit":
        classes = dict(h=qc.hadamard, cnot=qc.cnot, x=qc.Xgate, y=qc.Ygate, z=qc.Zgate)
        value, gates = _circuit(case, seed)
        start = q.it_t()
        start.upload(HostState.from_objects([bytes(value)]))
        return dict(case=case, start=start, pair=(q.it_t(), q.it_t()), gates=[classes[g[0]](*g[1:]) for g in gates])
    if kind == "walk":
        left, right, mag = _walk_state(case, seed)
        n = case["nodes"]
        one = np.frombuffer(qcgd.make_graph(n), np.uint8)
        wide = (one.size + 7) // 8 * 8
        obj = np.zeros((left.size, wide), np.uint8)
        obj[:, :one.size] = one
        at = np.arange(n, dtype=np.uint64)
        obj[:, 2:2 + n] = (left[:, None] >> at) & np.uint64(1)
        obj[:, 2 + n:2 + 2 * n] = (right[:, None] >> at) & np.uint64(1)
        start = q.it_t()
        start.upload(HostState(obj.reshape(-1), np.arange(left.size + 1, dtype=np.uint64) * np.uint64(wide),
                               np.full(left.size, one.size, np.uint32), mag))
        return dict(case=case, start=start, out=q.it_t(), rule=qcgd.coin(*_walk_angles(seed)))
    if kind == "step":
        ctx = _context(case["chunk_log2"])
        rules = _rules(_angles(rng))
        state = dict(case=case, start=_grown(case, rules, ctx), out=q.it_t(ctx=ctx),
                     rule=rules[0 if case["rule"] == "split_merge" else 1], seed=seed)
        return _outputs(state, state["start"], case["cap"] * 80 * max(case["nodes"], 8))
    if kind == "batch":
        graphs = random.Random(case["graph"])
        sizes = [graphs.randint(case["lo"], case["hi"]) for _ in range(case["instances"])]
        rules = [_rules(_angles(rng)) for _ in sizes]
        rules = [[r[0] for r in rules], [r[1] for r in rules]]
        a = qb.batch_t.from_states([HostState.from_objects([_graph(n, graphs)]) for n in sizes])
        b, c = qb.batch_t(), qb.batch_t()
        for _ in range(2):
            qb.apply_modifier(a, qcgd.step)
            for r in rules:
                qb.simulate_batched(a, r, b, case["cap"])
                a, b = b, a
        qb.apply_modifier(a, qcgd.step)
        state = dict(case=case, start=a, mid=b, out=c, rules=rules)
        return _outputs(state, a.state, case["instances"] * case["cap"] * 80 * max(case["hi"], 8))
    start = q.it_t()
    start.upload(HostState.from_objects([_graph(case["nodes"], random.Random(case["graph"]))]))
    return dict(case=case, start=start, program=adj.qcgd_program(case["iterations"], case["cap"]),
                params=np.array(_angles(rng)))


# -- one pass -------------------------------------------------------------
class _DeviceArray:
    """A device array of the library as torch sees it; keeps its owner."""

    def __init__(self, owner, pointer, count, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=(count,), typestr=typestr, data=(pointer or 0, False), version=2)


def _state(it, state):
    """The resulting state's own arrays, and its object bytes (of varying
    number: in the program's own tensor)."""
    obj, begin, size, mag = (ctypes.c_void_p() for _ in range(4))
    check(lib().qd_state_device_ptrs(it.handle, ctypes.byref(obj), ctypes.byref(begin), ctypes.byref(size),
                                     ctypes.byref(mag)), "qd_state_device_ptrs")
    n, nbytes, total = it.info()
    objects = torch.as_tensor(_DeviceArray(it, obj.value, nbytes, "|u1"), device="cuda")
    if "bytes" in state:
        with torch.cuda.stream(state["stream"]):
            state["bytes"][:nbytes].copy_(objects)
        objects = state["bytes"]
    return dict(objects=objects,
                begin=torch.as_tensor(_DeviceArray(it, begin.value, n + 1, "<i8"), device="cuda"),
                size=torch.as_tensor(_DeviceArray(it, size.value, n, "<i4"), device="cuda"),
                mag=torch.as_tensor(_DeviceArray(it, mag.value, 2 * n, "<f8"), device="cuda"),
                total=np.array([total]))


_COUNTS = ("num_candidates", "num_unique", "num_survivors")


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "loop":
        cap = case["cap"] or UNLIMITED
        src, (a, b) = state["start"], state["pair"]
        nodes, counts = [], []
        for _ in range(case["iterations"]):
            for rule, dst in zip(state["rules"], (a, b)):
                st = q.simulate(src, rule, dst, None, cap)
                counts += [st[k] for k in _COUNTS]
                src = dst
            nodes.append(adj.average_value(src, adj.OBS_NUM_NODES))
            q.simulate(src, qcgd.step)
        return dict(_state(src, state), nodes=np.array(nodes), counts=np.array(counts))
    if kind == "circuit":
        src, (a, b) = state["start"], state["pair"]
        for gate in state["gates"]:
            if gate.is_modifier:
                q.simulate(src, gate)
            else:
                q.simulate(src, gate, a, None, UNLIMITED)
                src, a, b = a, b, a
        return _state(src, state)
    if kind in ("walk", "step"):
        q.simple_truncation, q.truncation_seed = not case.get("probabilistic", False), state.get("seed", 0)
        st = q.simulate(state["start"], state["rule"], state["out"], None, case.get("cap", UNLIMITED))
        q.simple_truncation, q.truncation_seed = True, 0
        return dict(_state(state["out"], state), counts=np.array([st[k] for k in _COUNTS]))
    if kind == "batch":
        got = []
        for src, rules, dst in ((state["start"], state["rules"][0], state["mid"]),
                                (state["mid"], state["rules"][1], state["out"])):
            stats = qb.simulate_batched(src, rules, dst, case["cap"])
            got.append(dict(counts=np.array([[s[k] for k in _COUNTS] for s in stats]),
                            totals=np.array([s["total_proba"] for s in stats])))
        return dict(_state(state["out"].state, state), calls=got, seg=state["out"].seg.astype(np.int64))
    value, grad = adj.gradient(state["program"], state["params"], state["start"], adj.OBS_PARTICLES, 0,
                               case["checkpoint"])
    return dict(value=np.array([value]), grad=grad)


# -- what a pass cannot do without ----------------------------------------
def _children(rule, nodes):
    """Mean number of children of a grown state's parent (fitted to runs of
    6 to 16 nodes)."""
    return {"split_merge": 1.46, "erase_create": 1.53}[rule] ** nodes


def _step_work(parents, children, size, out, decisions):
    """Parents and survivors moved once, with 28 bytes of magnitude, offset
    and size each; per candidate a complex product per decision, its sum and
    its norm."""
    return parents * (size + 28) + out * (size + 28), parents * children * (6 * decisions + 5)


def work(case):
    kind, nbytes, flops = case["kind"], 0.0, 0.0
    n = case.get("nodes", 0)

    def add(p, children, size, out, decisions, times=1):
        nonlocal nbytes, flops
        b, f = _step_work(p, children, size, out, decisions)
        nbytes += times * b
        flops += times * f

    def loop(nodes, iterations, cap, times=1):
        p = 1.0
        for _ in range(iterations):
            for rule in ("split_merge", "erase_create"):
                c = _children(rule, nodes)
                out = min(p * c, cap)
                add(p, c, 44 * nodes, out, nodes / 2, times)
                p = out

    if kind == "loop":
        loop(n, case["iterations"], case["cap"] or math.inf)
    elif kind == "circuit":
        for k in range(case["gates"]):
            p = 2 ** min(k, case["qubits"])
            add(p, 2, case["qubits"], 2 ** min(k + 1, case["qubits"]), 1)
    elif kind == "walk":
        kids = 2.0 ** (case["particles"] * (1 - case["particles"] / (2 * n)))
        add(case["parents"], kids, 4 + 20 * n, case["parents"] * kids, case["particles"])
    elif kind == "step":
        add(case["parents"], _children(case["rule"], n), 44 * n, case["cap"], n / 2)
    elif kind == "batch":
        mid = (case["lo"] + case["hi"]) / 2
        for rule in ("split_merge", "erase_create"):
            add(case["cap"] * case["instances"], _children(rule, mid), 44 * mid, case["cap"] * case["instances"],
                mid / 2)
    else:  # forward, recomputation of all but the last segment, and the adjoint
        loop(n, case["iterations"], case["cap"], 3)
    return dict(bytes=float(nbytes), flops=float(flops))


# -- the same in plain numpy and Python -----------------------------------
def _polar(rho, phi):
    return complex(rho * math.cos(phi), rho * math.sin(phi))


def _coefficients(theta, phi, xi=0.0):
    """(done, not done): of an operation and of its inverse."""
    do, no = _polar(math.sin(theta), phi), _polar(math.cos(theta), xi)
    return {False: (do, no), True: (do.conjugate(), -no.conjugate())}


def _exact_walk(case, seed):
    left, right, mag = _walk_state(case, seed)
    coef = _coefficients(*_walk_angles(seed))
    n = case["nodes"]
    place = np.arange(n, dtype=np.uint64)
    can = ((left ^ right)[:, None] >> place) & np.uint64(1) != 0
    kids = can.sum(1)
    first = np.concatenate([[0], np.cumsum(1 << kids)])
    L, R = np.empty(first[-1], np.uint64), np.empty(first[-1], np.uint64)
    M = np.empty(first[-1], np.complex128)
    for k in np.unique(kids):
        rows = np.nonzero(kids == k)[0]
        where = np.nonzero(can[rows])[1].reshape(rows.size, k).astype(np.uint64)
        for child in range(1 << int(k)):
            l, r, m = left[rows].copy(), right[rows].copy(), mag[rows].copy()
            for d in range(int(k)):
                conj = (left[rows] >> where[:, d]) & np.uint64(1) != 0
                done = child >> d & 1
                m *= np.where(conj, coef[True][1 - done], coef[False][1 - done])
                if done:
                    l ^= np.uint64(1) << where[:, d]
                    r ^= np.uint64(1) << where[:, d]
            L[first[rows] + child], R[first[rows] + child], M[first[rows] + child] = l, r, m
    order = np.lexsort((np.arange(L.size), R, L))
    start = np.ones(L.size, bool)
    start[1:] = (L[order][1:] != L[order][:-1]) | (R[order][1:] != R[order][:-1])
    at = np.nonzero(start)[0]
    total = np.add.reduceat(M[order], at)
    rep = order[at]  # the group's smallest candidate: the order is by candidate within a group
    norm = np.abs(total) ** 2
    keep = np.nonzero(norm > 1e-30)[0]
    keep = keep[np.argsort(rep[keep])]
    s = norm[keep].sum()
    out = (total[keep] / np.sqrt(s)).view(np.float64)
    return dict(objects=None, begin=None, size=None, mag=out, total=np.array([s]), counts=None)


def _exact_circuit(case, seed):
    value, gates = _circuit(case, seed)
    keys = np.array([sum(v << i for i, v in enumerate(value))])
    mag = np.ones(1, np.complex128)
    s = 1.0
    for name, *bits in gates:
        one = keys >> bits[-1] & 1
        if name == "h":
            c = 1 / math.sqrt(2)
            keys = np.stack([keys ^ (1 << bits[0]), keys], 1).reshape(-1)
            mag = np.stack([mag * c, mag * np.where(one, -c, c)], 1).reshape(-1)
            keys, at, group = np.unique(keys, return_index=True, return_inverse=True)
            mag = np.bincount(group, mag.real) + 1j * np.bincount(group, mag.imag)
            order = np.argsort(at)
            order = order[np.abs(mag[order]) ** 2 > 1e-30]
            keys, mag = keys[order], mag[order]
            s = np.sum(np.abs(mag) ** 2)
            mag = mag / np.sqrt(s)
        elif name == "cnot":
            keys = keys ^ ((keys >> bits[0] & 1) << bits[1])
        else:
            if name == "y":
                mag = mag * 1j
            if name != "x":
                mag = np.where(one, -mag, mag)
            keys = keys ^ (1 << bits[0])
    return dict(objects=None, begin=None, size=None, mag=mag.view(np.float64), total=np.array([s]))


# a node's name as a tree: an element is its number, the halves of a split are
# ("l", tree) and ("r", tree), a merged name is the pair (tree, tree)
def _is_pair(t):
    return isinstance(t, tuple) and t[0] not in ("l", "r")


def _half(t, side):
    return t[0 if side == "l" else 1] if _is_pair(t) else (side, t)


def _merged(a, b):
    if isinstance(a, tuple) and isinstance(b, tuple) and a[0] == "l" and b[0] == "r" and a[1] == b[1]:
        return a[1]
    return (a, b)


def _has_zero(t):
    """Whether the most left part of element 0 lies in the name."""
    if not isinstance(t, tuple):
        return t == 0
    return t[0] == "l" and _has_zero(t[1]) if not _is_pair(t) else _has_zero(t[0]) or _has_zero(t[1])


def _split_merge_children(graph, coef):
    left, right, names = graph
    n = len(names)
    split = [left[i] and right[i] for i in range(n)]
    merge = [i + 1 < n and not split[i] and left[i] and right[i + 1] and not left[i + 1] for i in range(n)]
    last = n > 1 and not split[0] and right[0] and left[n - 1] and not right[n - 1]
    decisions = int(last) + sum(split[i] or merge[i] for i in range(n))
    for child in range(1 << decisions):
        bits, mag, nodes, late = child, 1 + 0j, [], []

        def choose(inverse):
            nonlocal bits, mag
            done = bits & 1
            bits >>= 1
            mag *= coef[inverse][1 - done]
            return done

        begin, end = 0, n
        if last and choose(True):
            nodes.append((True, True, _merged(names[n - 1], names[0])))
            begin, end = 1, n - 1
        i = begin
        while i < end:
            if split[i] and choose(False):
                a, b = _half(names[i], "l"), _half(names[i], "r")
                first = (True, False, a)
                if i == 0 and _is_pair(names[0]) and not _has_zero(names[0][0]):
                    late = [first]  # the half without element 0's start goes round to the end
                else:
                    nodes.append(first)
                nodes.append((False, True, b))
            elif merge[i] and choose(True):
                nodes.append((True, True, _merged(names[i], names[i + 1])))
                i += 1
            else:
                nodes.append((left[i], right[i], names[i]))
            i += 1
        yield tuple(zip(*(nodes + late))), mag


def _erase_create_children(graph, coef):
    left, right, names = graph
    where = [i for i in range(len(names)) if left[i] == right[i]]
    for child in range(1 << len(where)):
        l, r, mag = list(left), list(right), 1 + 0j
        for d, i in enumerate(where):
            done = child >> d & 1
            mag *= coef[left[i]][1 - done]
            if done:
                l[i], r[i] = not l[i], not r[i]
        yield (tuple(l), tuple(r), names), mag


def _exact_loop(case, seed):
    a = _angles(random.Random(seed))
    n = case["nodes"]
    left, right = _particles(n, random.Random(case["graph"]))
    state = {(tuple(map(bool, left)), tuple(map(bool, right)), tuple(range(n))): 1 + 0j}
    rules = [(_split_merge_children, _coefficients(a[0], a[1])), (_erase_create_children, _coefficients(a[2], a[3]))]
    nodes, s = [], 1.0
    for _ in range(case["iterations"]):
        for children, coef in rules:
            new = {}
            for graph, mag in state.items():  # insertion order is the order of first candidates
                for child, factor in children(graph, coef):
                    new[child] = new.get(child, 0j) + mag * factor
            new = {g: m for g, m in new.items() if abs(m) ** 2 > 1e-30}
            s = math.fsum(abs(m) ** 2 for m in new.values())
            state = {g: m / math.sqrt(s) for g, m in new.items()}
        nodes.append(math.fsum(len(g[2]) * abs(m) ** 2 for g, m in state.items()))
        state = {(g[0][1:] + g[0][:1], g[1][-1:] + g[1][:-1], g[2]): m for g, m in state.items()}
    mag = np.array(list(state.values()), np.complex128).view(np.float64)
    return dict(objects=None, begin=None, size=None, mag=mag, total=np.array([s]), nodes=np.array(nodes), counts=None)


def exact(case, seed):
    kind = case["kind"]
    if kind == "walk":
        return _exact_walk(case, seed)
    if kind == "circuit":
        return _exact_circuit(case, seed)
    if kind == "loop" and not case["cap"] and case["nodes"] <= 6:
        return _exact_loop(case, seed)
    # (truncated states hold ties and near ties, which rounding cuts one way
    # or the other: no value in another arithmetic)
    return None
