"""Kerma-estimator tallies whose images lie side by side for each voxel and are added to by pairs
of lanes: every combination of images, with and without room in LDS for the exchange, and after
a reset and a launch search, equals the oracle's."""
import numpy as np
import pytest

from oracle import oracle as O
from opengate_amd.transport import PhantomSpec, SourceSpec, TallySpec

from helpers import aligned_tally, centre, small_phantom, tables

pytestmark = pytest.mark.gpu


def _same(gpu, ref, counters, ref_counters):
    for k in ("histories", "steps", "deposits", "sq_evictions", "photo", "compton"):
        assert counters[k] == ref_counters[k], k
    for k in gpu:
        # FP64 sums in another order, as for the analog tallies
        assert np.max(np.abs(gpu[k] - ref[k])) <= 1e-9 * np.abs(ref[k]).max(), k


@pytest.mark.parametrize("launch", [{"block": 0}, {"block": 64, "grid": 3}])
@pytest.mark.parametrize("images", [{"edep2": False}, {}, {"dose": True}, {"dose2": True, "edep2": False},
                                    {"dose": True, "dose2": True, "counts": True}])
def test_images(engine, images, launch):
    T, ph = tables(e_max=0.21), small_phantom(24, 2.0)
    src = SourceSpec(pos_trans=centre(ph), energy=0.1405)
    tal = TallySpec(size=(20, 17, 11), spacing=(2.0, 2.5, 3.0), corner=(3.0, 1.0, 7.0), aligned=False, tle=True,
                    tle_energy_min=0.003, tle_energy_max=0.12, **images)
    engine.clear()
    engine.set_physics(T)
    sid = engine.add_simulation(ph, src, tal)
    print(f"[gpu case] TLE images {images} {launch}", flush=True)
    engine.run([3000], 1, **launch)
    engine.reset_tally(sid)
    c = engine.run([40_000], 21, **launch)
    before = engine.get_tally(sid)
    engine.autotune([2000])
    g = engine.get_tally(sid)
    r, rc = O.run(T, ph, src, tal, 40_000, 21)
    assert set(g) == {"edep", "edep2", "dose", "dose2", "counts"} & (
        {"edep"} | ({"edep2"} if images.get("edep2", True) else set()) | set(images) - {"edep2"})
    for k in g:
        assert np.array_equal(g[k], before[k])
    _same(g, r, c, rc)


def test_no_room_for_the_exchange(engine):
    from opengate_amd.physics import xs
    from opengate_amd.physics.materials import MaterialDatabase
    from opengate_amd.units import g4_units

    db = MaterialDatabase()
    names = ["G4_WATER", "G4_BONE_CORTICAL_ICRP"]
    nb1 = tables().n_buckets + 1
    m = 80000 // (4 * nb1)  # mu and majorant fill the 1024-thread budget but for less than 8 KiB
    for k in range(m - 2):
        db.add_material_weights(f"WATER_{k}", ["H", "O"], [0.111894, 0.888106],
                                (0.9 + 0.02 * k) * g4_units.g / g4_units.cm3)
        names.append(f"WATER_{k}")
    T = xs.build_tables([db.get(n) for n in names], 0.1405)
    lds1 = 4 * (m + 1) * (T.n_buckets + 1) + 8 * m
    assert 77_000 < lds1 < 84_000
    lab = np.random.default_rng(1).integers(0, m, size=(13, 11, 9)).astype(np.uint8)
    ph = PhantomSpec(lab, (2.0, 2.5, 3.0))
    src = SourceSpec(pos_trans=centre(ph), energy=0.1)
    tal = aligned_tally(ph, tle=True)
    engine.clear()
    engine.set_physics(T)
    sid = engine.add_simulation(ph, src, tal)
    print(f"[gpu case] TLE with {m} materials, block 1024", flush=True)
    c = engine.run([50_000], 4, block=1024)
    r, rc = O.run(T, ph, src, tal, 50_000, 4)
    _same(engine.get_tally(sid), r, c, rc)
