"""Launches of several simulations whose point sources add into tally copies: the images equal those
of the same histories run in pieces too short for copies, for every place and kind of neighbour."""
import numpy as np
import pytest

from opengate_amd.transport import SourceSpec, TallySpec

from helpers import centre, small_phantom, tables

pytestmark = pytest.mark.gpu


# histories of each simulation; 500000 of a simulation among several are the line for copies
@pytest.mark.parametrize("n", [[600000, 500000], [499999, 700000, 0, 600000], [1, 520000, 3000]])
def test_batched_copies(engine, n):
    print(f"[gpu case] tally copies in a launch of {n}", flush=True)
    T, ph = tables(), small_phantom(24, 2.0)
    point = SourceSpec(pos_trans=centre(ph), energy=0.1405)
    box = SourceSpec(pos_type="box", pos_param=(4.0, 4.0, 4.0), pos_trans=centre(ph), energy=0.1405)
    tallies = [TallySpec(size=(3, 5, 7), spacing=(40.0 / 3, 8.0, 40.0 / 7), corner=(3.0, 1.0, 7.0), aligned=False,
                         dose=True, dose2=True, counts=True),
               TallySpec(size=(24, 24, 24), spacing=(2.0,) * 3),
               TallySpec(size=(20, 17, 11), spacing=(2.0, 40.0 / 17, 40.0 / 11), aligned=False, edep2=False),
               TallySpec(size=(24, 24, 24), spacing=(2.0,) * 3)]
    engine.clear()
    engine.set_physics(T)
    for k in range(len(n)):
        engine.add_simulation(ph, box if k == 3 else point, tallies[k])
    c = [engine.run(n, 21), engine.run(n, 22)]  # the copies are clear again behind a run
    got = [engine.get_tally(k) for k in range(len(n))]
    for k in range(len(n)):
        engine.reset_tally(k)
    ref = [{"histories": 0, "steps": 0, "deposits": 0} for _ in c]
    for seed, r in zip((21, 22), ref):
        for lo in range(0, max(n), 300000):
            part = engine.run([max(0, min(300000, v - lo)) for v in n], seed, first_history=[lo] * len(n))
            for name in r:
                r[name] += part[name]
    for a, r in zip(c, ref):
        assert all(a[name] == r[name] for name in r)
    for k in range(len(n)):
        want = engine.get_tally(k)
        assert (want["edep"].max() > 0) == (n[k] > 0)
        for name in want:
            assert np.max(np.abs(got[k][name] - want[name])) <= 1e-9 * max(np.abs(want[name]).max(), 1e-300), (k, name)
