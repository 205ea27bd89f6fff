"""The transport's work queue: every split of a run over workgroups and chunks (fewer
workgroups than queues, chunks of one history, ragged ends, several simulations) runs each
history exactly once, with the counters and tallies of the automatic launch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

INTS = ("histories", "steps", "deposits", "compton", "rayleigh", "photo", "escaped", "cut_kills", "sq_evictions")


def _check(a, b, ta, tb):
    assert all(a[k] == b[k] for k in INTS), [(k, a[k], b[k]) for k in INTS if a[k] != b[k]]
    for k in ("e_deposited", "e_escaped"):
        assert abs(a[k] - b[k]) <= 1e-9 * abs(a[k])
    for x, y in zip(ta, tb):
        # FP64 sums in another order
        assert np.max(np.abs(x["edep"] - y["edep"])) <= 1e-9 * max(x["edep"].max(), 1e-300)


@pytest.mark.parametrize("n,grid,chunk,block", [(1, 0, 1, 0), (63, 1, 7, 256), (4097, 3, 64, 256), (4097, 9, 1, 64),
                                                (70001, 0, 16, 256), (70001, 7, 4096, 1024), (300001, 0, 64, 1024),
                                                (300001, 17, 100, 192)])
def test_single(n, grid, chunk, block):
    from opengate_amd import workloads
    from opengate_amd.transport import GpuEngine

    print(f"[gpu case] queue n={n} grid={grid} chunk={chunk} block={block}", flush=True)
    tables, ph, src, tal, _ = workloads.water64()
    eng = GpuEngine(0)
    eng.set_physics(tables)
    eng.add_simulation(ph, src, tal)
    a = eng.run([n], 3)
    ta = [eng.get_tally(0)]
    eng.reset_tally(0)
    b = eng.run([n], 3, grid=grid, chunk=chunk, block=block)
    assert b["histories"] == n
    _check(a, b, ta, [eng.get_tally(0)])
    eng.close()


@pytest.mark.parametrize("grid,chunk", [(0, 0), (5, 33), (40, 256)])
def test_batched(grid, chunk):
    from opengate_amd import workloads
    from opengate_amd.transport import GpuEngine

    print(f"[gpu case] queue batched grid={grid} chunk={chunk}", flush=True)
    tables, ph, src, tal, _ = workloads.water64()
    n = [5000, 0, 1, 777]
    eng = GpuEngine(0)
    eng.set_physics(tables)
    for _ in n:
        eng.add_simulation(ph, src, tal)
    a = eng.run(n, 3, chunk=64)
    ta = [eng.get_tally(k) for k in range(len(n))]
    for k in range(len(n)):
        eng.reset_tally(k)
    b = eng.run(n, 3, grid=grid, chunk=chunk)
    assert b["histories"] == sum(n)
    _check(a, b, ta, [eng.get_tally(k) for k in range(len(n))])
    eng.close()
