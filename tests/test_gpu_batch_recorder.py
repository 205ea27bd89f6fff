"""Several simulations that record in one launch: the automatic chunks (large, so that the
simulations' recorders are used side by side) give the records, tallies and counters of small ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [[1500000, 0, 2000000, 1700000], [3000, 1, 70000]])
def test_records_of_any_chunk(n):
    from opengate_amd import workloads
    from opengate_amd.transport import GpuEngine, PhantomSpec, SourceSpec, TallySpec

    print(f"[gpu case] recorders of a launch of {n}", flush=True)
    eng = GpuEngine(0)
    eng.set_physics(workloads.water64()[0])
    for k, h in enumerate(n):
        eng.add_simulation(PhantomSpec(np.zeros((16, 16, 16), np.uint8), (4.0,) * 3),
                           SourceSpec(pos_type="box", pos_param=(20.0,) * 3, pos_trans=(32.0,) * 3, energy=0.1405),
                           TallySpec(size=(16,) * 3, spacing=(4.0,) * 3, record_face=6 if k != 1 else -1,
                                     record_capacity=h if k != 1 else 0))
    out = []
    for chunk in (0, 64):
        for k in range(len(n)):
            eng.reset_tally(k)
            if k != 1:
                eng.reset_phsp(k)
        c = eng.run(n, 5, chunk=chunk)
        rec = []
        for k in range(len(n)):
            if k != 1:
                r = np.stack(eng.get_phsp(k)[0]) if n[k] else np.zeros((8, 0))
                rec.append(r[:, np.lexsort(r)])
        out.append((c, rec, [eng.get_tally(k)["edep"] for k in range(len(n))]))
    (ca, ra, ta), (cb, rb, tb) = out
    assert ca["histories"] == sum(n) and ca["recorded"] > 0
    assert all(ca[k] == cb[k] for k in ("histories", "steps", "deposits", "recorded", "escaped"))
    for a, b in zip(ra, rb):
        assert np.array_equal(a, b)
    for a, b in zip(ta, tb):
        assert np.max(np.abs(a - b)) <= 1e-9 * max(b.max(), 1e-300)
    eng.close()
