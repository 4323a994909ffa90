"""Survivors whose bytes pass 2^32 within one tile of the order (4096
candidates): every child where it belongs, bit for bit."""
import numpy as np
import pytest

import quids_amd as q
from oracle import oracle as orc
from quids_amd.rules import quantum_computer as qc
from quids_amd.state import HostState

pytestmark = pytest.mark.gpu


def _registers(n, width, size):
    """n registers of `size` qubits, the last ones beyond `width` all 0: the
    one that the gate acts on, a number, and random ones."""
    rng = np.random.default_rng(7)
    obj = np.zeros((n, size), np.uint8)
    obj[:, :width] = rng.integers(0, 2, (n, width))
    for k in range(12):
        obj[:, 1 + k] = (np.arange(n) >> k) & 1
    mag = rng.normal(size=n) + 1j * rng.normal(size=n)
    return HostState(obj.reshape(-1), np.arange(n + 1, dtype=np.uint64) * np.uint64(size),
                     np.full(n, size, np.uint32), mag / np.linalg.norm(mag))


def test_a_tile_of_more_than_4_gib():
    n, width, size = 2048, 64, (1 << 20) + 64
    a, b = q.it_t(), q.it_t()
    a.upload(_registers(n, width, size))
    st = q.simulate(a, qc.hadamard(0), b, None, q.UINT64_MAX)
    got = b.download()
    a.close()
    b.close()
    # the same registers, short: the children's bytes and magnitudes
    ref, ost = orc.simulate(_registers(n, width, width), qc.hadamard(0))
    assert st["num_unique"] == ost["num_unique"] == 2 * n
    assert np.array_equal(got.object_begin, np.arange(2 * n + 1, dtype=np.uint64) * np.uint64(size))
    assert np.all(got.object_size == size)
    rows = got.objects.reshape(2 * n, size)
    assert np.array_equal(rows[:, :width], ref.objects.reshape(2 * n, width))
    assert not rows[:, width:].any()
    assert np.array_equal(got.magnitude, ref.magnitude)
