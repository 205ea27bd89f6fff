"""Runs that add into several copies of small tallies (a point source inside the phantom, many
histories): the folded images equal the oracle's, run after run."""
import numpy as np
import pytest

from oracle import oracle as O
from opengate_amd.transport import SourceSpec, TallySpec

from helpers import centre, small_phantom, tables

pytestmark = pytest.mark.gpu


# 4 histories a value are the line: 3 x 5 x 7 voxels and 2 images 840, 20 x 17 x 11 and 5 images 74800
@pytest.mark.parametrize("size,images,tle,n", [((3, 5, 7), {}, False, 839), ((3, 5, 7), {}, False, 840),
                                               ((3, 5, 7), {}, True, 30000), ((1, 1, 1), {"edep2": False}, False, 5000),
                                               ((20, 17, 11), {"dose": True, "dose2": True, "counts": True}, False, 74800),
                                               ((20, 17, 11), {"dose": True, "dose2": True, "counts": True}, True, 80000)])
def test_folded_runs(engine, size, images, tle, n):
    T, ph = tables(), small_phantom(24, 2.0)
    src = SourceSpec(pos_trans=centre(ph), energy=0.1405)
    tal = TallySpec(size=size, spacing=tuple(40.0 / s for s in size), corner=(3.0, 1.0, 7.0), aligned=False, tle=tle,
                    **images)
    engine.clear()
    engine.set_physics(T)
    sid = engine.add_simulation(ph, src, tal)
    print(f"[gpu case] tally copies {size} {images} tle={tle} n={n}", flush=True)
    engine.run([n], 1)
    engine.reset_tally(sid)
    c = [engine.run([n], 21), engine.run([n], 22)]
    g = engine.get_tally(sid)
    runs = [O.run(T, ph, src, tal, n, seed) for seed in (21, 22)]
    for a, (_, b) in zip(c, runs):
        assert all(a[k] == b[k] for k in ("histories", "steps", "deposits", "sq_evictions", "escaped"))
    for k in g:
        ref = sum(r[k] for r, _ in runs)
        assert np.max(np.abs(g[k] - ref)) <= 1e-9 * np.abs(ref).max(), k


def test_point_outside_and_other_sources(engine):
    T, ph = tables(), small_phantom(12, 4.0)
    c = centre(ph)
    for src in (SourceSpec(pos_trans=(c[0], c[1], -5.0), energy=0.1405),
                SourceSpec(pos_type="box", pos_param=(4.0, 4.0, 4.0), pos_trans=c, energy=0.1405)):
        tal = TallySpec(size=(4, 4, 4), spacing=(12.0, 12.0, 12.0))
        tal.aligned = False
        engine.clear()
        engine.set_physics(T)
        sid = engine.add_simulation(ph, src, tal)
        print(f"[gpu case] no tally copies {src.pos_type}", flush=True)
        engine.run([20000], 5)
        g = engine.get_tally(sid)
        r, _ = O.run(T, ph, src, tal, 20000, 5)
        assert np.max(np.abs(g["edep"] - r["edep"])) <= 1e-9 * r["edep"].max()
