"""The radix passes that a step reports are those that its dedup used: the
layouts of device-driven steps and of host-driven ones (qd_tuning.eager_select)
differ at these sizes."""
import numpy as np
import pytest

import quids_amd as q
from quids_amd.rules import quantum_computer as qc
from quids_amd.state import HostState

pytestmark = pytest.mark.gpu


# candidates 2n: one bucket or two; one pass or two; and two where the host
# takes up the select (more equal keys than one block takes)
@pytest.mark.parametrize("n,cap,device,host", [(50, q.UINT64_MAX, 0, 0), (100, q.UINT64_MAX, 1, 0),
                                               (65000, q.UINT64_MAX, 2, 1), (65000, 65000, 2, 1)])
def test_dedup_levels(n, cap, device, host):
    obj = np.zeros((n, 8), np.uint8)
    for k in range(3):
        obj[:, 1 + k] = (np.arange(n) >> (8 * k)) & 0xFF
    hs = HostState(obj.reshape(-1), np.arange(n + 1, dtype=np.uint64) * np.uint64(8), np.full(n, 4, np.uint32),
                   np.full(n, n ** -0.5 + 0j))
    ctx = q.default_context()
    old = ctx.get_tuning()
    a, b = q.it_t(), q.it_t()
    a.upload(hs)
    try:
        for eager, levels in ((0, device), (1, host)):
            ctx.set_tuning(eager_select=eager)
            assert q.simulate(a, qc.hadamard(0), b, None, cap)["dedup_levels"] == levels, eager
    finally:
        ctx.set_tuning(eager_select=old["eager_select"])
    a.close()
    b.close()
