"""Tallies fetched into ordinary host arrays (staged blocks, one thread or several) equal, bit
for bit, the copy that the runtime makes straight into pinned memory."""
import ctypes as C

import numpy as np
import pytest
import torch

from opengate_amd import _abi as A

pytestmark = pytest.mark.gpu


# block of 131072 doubles: below, at and over one block; two threads; all of them, ragged
@pytest.mark.parametrize("n", [1, 131071, 131072, 131073, 393217, 1048577, 6291456, 8388611])
def test_tally_equals_pinned_copy(n):
    from opengate_amd import workloads
    from opengate_amd.transport import GpuEngine, TallySpec

    print(f"[gpu case] host copy n={n}", flush=True)
    tables, ph, src, _, _ = workloads.water64()
    tal = TallySpec(size=(n, 1, 1), spacing=(128.0 / n, 128.0, 128.0), aligned=False)
    eng = GpuEngine(0)
    eng.set_physics(tables)
    eng.add_simulation(ph, src, tal)
    eng.run([50000], 5)
    pinned = [torch.empty(n, dtype=torch.float64, pin_memory=True) for _ in range(2)]
    p = [C.cast(C.c_void_p(t.data_ptr()), A.DP) for t in pinned]
    eng._check(eng.lib.gh_get_tally(eng.ctx, 0, p[0], p[1], A.DP(), A.DP(), A.DP()), "gh_get_tally")
    got = eng.get_tally(0)
    assert pinned[0].sum() > 0
    for t, k in zip(pinned, ("edep", "edep2")):
        assert np.array_equal(t.numpy(), got[k].reshape(-1))
    eng.close()


def test_contexts_in_threads():
    # staging blocks change hands between contexts: copies of several host threads at once
    import threading

    from opengate_amd import workloads
    from opengate_amd.transport import GpuEngine, TallySpec

    print("[gpu case] host copy of three contexts at once", flush=True)
    tables, ph, src, _, _ = workloads.water64()
    engines, want, bad = [], [], []
    for n in (1000, 400000, 3000000):
        eng = GpuEngine(0)
        eng.set_physics(tables)
        eng.add_simulation(ph, src, TallySpec(size=(n, 1, 1), spacing=(128.0 / n, 128.0, 128.0), aligned=False))
        eng.run([20000], 5)
        engines.append(eng)
        want.append(eng.get_tally(0)["edep"])

    def fetch(k):
        for _ in range(5):
            if not np.array_equal(engines[k].get_tally(0)["edep"], want[k]):
                bad.append(k)

    threads = [threading.Thread(target=fetch, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    for eng in engines:
        eng.close()
