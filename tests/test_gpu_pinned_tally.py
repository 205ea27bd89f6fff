"""Tallies into pinned destinations anywhere in their allocation (its start, inside, up to its last
byte): the values of an ordinary fetch and nothing written around them."""
import ctypes as C

import numpy as np
import pytest
import torch

from opengate_amd import _abi as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 1000, 300001])
def test_places_in_a_pinned_allocation(n):
    from opengate_amd import workloads
    from opengate_amd.transport import GpuEngine, TallySpec

    print(f"[gpu case] pinned tally n={n}", flush=True)
    tables, ph, src, _, _ = workloads.water64()
    eng = GpuEngine(0)
    eng.set_physics(tables)
    eng.add_simulation(ph, src, TallySpec(size=(n, 1, 1), spacing=(128.0 / n, 128.0, 128.0), aligned=False))
    eng.run([50000], 5)
    want = eng.get_tally(0)
    for before, after in ((0, 0), (0, 700), (513, 700), (513, 0)):
        mem = [torch.full((before + n + after,), -1.0, dtype=torch.float64, pin_memory=True) for _ in range(2)]
        p = [C.cast(C.c_void_p(t.data_ptr() + 8 * before), A.DP) for t in mem]
        eng._check(eng.lib.gh_get_tally(eng.ctx, 0, p[0], p[1], A.DP(), A.DP(), A.DP()), "gh_get_tally")
        for t, k in zip(mem, ("edep", "edep2")):
            t = t.numpy()
            assert np.array_equal(t[before:before + n], want[k].reshape(-1))
            assert np.all(t[:before] == -1) and np.all(t[before + n:] == -1)
    eng.close()
