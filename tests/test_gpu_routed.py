"""The routed step's joined launches (fk_routed.h) on the GPU: every value
that the launches they replace store, bit for bit the oracle's CPU target's
(which runs those launches one by one), at one to four ranks, experts at and
past a wavefront's rows, widths that leave lanes' packs over, and each type
of table; eager and through a graph."""

import numpy as np
import pytest

from furykernel_amd.engine import Engine
from furykernel_amd.lower import routed_fusions
from routed_cases import CASES, case_id, cpu_values, lowered_case, state_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", CASES, ids=case_id)
def test_joined_launches_bit_exact(device, kernels, case):
    low = lowered_case(case)
    weights, x = state_of(case)
    want = cpu_values(low, case, weights, x)
    print(f"routed {case_id(case)}: {[L.entry for _, _, L in routed_fusions(low)]}", flush=True)
    eng = Engine(device, kernels, low)
    try:
        eng.write_weights({k: v.ravel() for k, v in weights.items()})
        eng.write("value:x", x)
        graph = None
        for how in ("eager", "graph", "graph"):
            for name in want:
                eng.zero(name)
            if how == "eager":
                eng.enqueue()
            else:
                graph = graph or eng.capture()
                graph.replay()
            device.sync()
            bad = [n for n, v in want.items() if not np.array_equal(eng.read(n).view(np.uint32), v.view(np.uint32))]
            assert bad == [], how
        # the same launches one by one
        for name in want:
            eng.zero(name)
        for i in range(len(low.launches)):
            eng.enqueue(only=[i])
        device.sync()
        assert [n for n, v in want.items() if not np.array_equal(eng.read(n).view(np.uint32), v.view(np.uint32))] == []
        graph.destroy()
    finally:
        eng.close()
