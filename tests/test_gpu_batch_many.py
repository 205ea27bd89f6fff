"""Launches of many simulations, some without histories: a chunk of the work queue finds its
simulation, whatever the chunk size. Every simulation's tally equals that of a launch in which only
it has histories (its random streams are keyed by its place)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_sims,chunk,grid", [(2, 0, 0), (65, 0, 0), (65, 7, 3), (300, 64, 0), (300, 1, 64)])
def test_chunks_find_their_simulation(n_sims, chunk, grid):
    from opengate_amd import workloads
    from opengate_amd.transport import GpuEngine, PhantomSpec, SourceSpec, TallySpec

    print(f"[gpu case] {n_sims} simulations chunk={chunk} grid={grid}", flush=True)
    tables = workloads.water64()[0]
    g = np.random.default_rng(n_sims)
    n = g.integers(1, 400, n_sims)
    n[g.random(n_sims) < 0.3] = 0
    n[-1] = 129
    n = [int(v) for v in n]
    eng = GpuEngine(0)
    eng.set_physics(tables)
    for k in range(n_sims):
        eng.add_simulation(PhantomSpec(np.zeros((8, 8, 8), np.uint8), (10.0,) * 3),
                           SourceSpec(pos_trans=(40.0,) * 3, energy=0.1405),
                           TallySpec(size=(8, 8, 8), spacing=(10.0,) * 3))
    c = eng.run(n, 11, chunk=chunk, grid=grid)
    assert c["histories"] == sum(n)
    got = [eng.get_tally(k)["edep"] for k in range(n_sims)]
    for k in [0, 1, n_sims // 2, n_sims - 2, n_sims - 1, *g.integers(0, n_sims, 10)]:
        eng.reset_tally(k)
        c = eng.run([v if i == k else 0 for i, v in enumerate(n)], 11)
        assert c["histories"] == n[k]
        want = eng.get_tally(k)["edep"]
        assert (got[k].max() > 0) == (n[k] > 0)
        assert np.max(np.abs(got[k] - want)) <= 1e-9 * max(want.max(), 1e-300)
    eng.close()
