"""Performance cases of the framework: what its users run, through the public entry points.

Each case is a plain dict; `prepare` makes what a program holds before the call (phantom,
tables, engine, network weights, recorded photons), `run` is one pass, `exact` the same
outputs in FP64 without the framework where such a value exists (a transport run follows the
framework's own random streams, so its tallies have none; its integer counters are exact).

Kinds:
  transport      GpuEngine.run of one simulation and the copy of its tally to the host
  batch          several simulations in one launch, every tally copied
  learned_dose   learned exit-plane source -> phase-space source -> ct phantom -> tally
  generate       photons of the learned exit-plane source (8 device arrays)
  project        photons that left a phantom -> SPECT projections by the learned response
  train          one training step of a dense network: forward, backward, Adam
  fit_exitplane  a short ExitPlaneGenerator.fit on recorded photons
  fit_response   a short ArfModel.fit on labelled photons
"""
import functools
import math
from pathlib import Path
from types import SimpleNamespace

import numpy as np
import torch

DEV = "cuda"
GENERATOR = "8-256-256-256-256-256-6"  # exit-plane generator
RESPONSE = "3-128-128-128-4"  # detector response
FOCAL = (32.0, 32.0, 142.5)  # point source of the collimator (its box frame, mm)
G_MAX, KNOTS = 5.5, 4096
COUNTERS = ("histories", "steps", "deposits", "compton", "rayleigh", "photo", "escaped", "world_interactions",
            "cut_kills", "sq_evictions", "recorded", "kn_rejections", "e_deposited", "e_outside_tally", "e_escaped",
            "e_world")


# ---------------------------------------------------------------------- cases
def listed():
    return [
        # a quick look at a simulation (a smoke run, a first test of a script): latency
        {"name": "water64_2e4", "kind": "transport", "phantom": "water", "nx": 64, "ny": 64, "nz": 64,
         "histories": 20_000, "tle": False},
        # the ordinary point-source dose run: 140.5 keV in a 64^3 water phantom, 1e6 histories
        {"name": "water64_1e6", "kind": "transport", "phantom": "water", "nx": 64, "ny": 64, "nz": 64,
         "histories": 1_000_000, "tle": False},
        # the CT dose production run: 256x256x128 voxels, 12 materials, 120 kVp cone
        {"name": "ct256_5e8", "kind": "transport", "phantom": "ct12", "nx": 256, "ny": 256, "nz": 128,
         "histories": 500_000_000, "tle": False},
        # CT dose with the Schneider conversion and the track-length estimator, odd image size
        {"name": "ct_schneider_tle_2e7", "kind": "transport", "phantom": "schneider", "nx": 201, "ny": 187, "nz": 93,
         "histories": 20_000_000, "tle": True},
        # a batch of small patient-like phantoms with volume sources in one launch
        {"name": "batch8_2e7", "kind": "batch", "n_sims": 8, "n_min": 64, "n_max": 128, "histories": 20_000_000},
        # dose of a learned source, end to end (generate, replay, tally)
        {"name": "learned_dose_2e7", "kind": "learned_dose", "photons": 20_000_000},
        # a few photons on request (an event loop that asks for small batches): latency
        {"name": "generate_1000", "kind": "generate", "photons": 1000},
        # a large phase-space in device memory
        {"name": "generate_1e7", "kind": "generate", "photons": 10_000_000},
        # projections of one run's escaping photons on 128 heads
        {"name": "project_1e6", "kind": "project", "photons": 1_000_000, "heads": 128, "squared": True},
        # one step of a training loop that computes its own loss, at the default batch
        {"name": "train_generator_16384", "kind": "train", "net": GENERATOR, "batch": 16384},
        # training the generator: features, quantile tables and a few steps
        {"name": "fit_exitplane", "kind": "fit_exitplane", "photons": 100_000, "steps": 6, "batch": 16384},
        # training the detector response on a small data set (batch = the whole ragged set)
        {"name": "fit_response_5003", "kind": "fit_response", "photons": 40_000, "steps": 6, "batch": 5003},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["transport", "transport", "transport", "batch", "learned_dose", "generate", "generate",
                       "project", "train", "train", "fit_exitplane", "fit_response"])
    c = {"kind": kind}
    if kind == "transport":
        c["phantom"] = rng.choice(["water", "ct12", "schneider"])
        if c["phantom"] == "water":
            n = rng.randint(40, 96)
            c.update(nx=n, ny=n + rng.randint(0, 9), nz=n + rng.randint(0, 9))
        else:
            c.update(nx=rng.randint(96, 256), ny=rng.randint(96, 256), nz=rng.randint(40, 128))
        c.update(histories=_log(rng, 20_000, 150_000_000), tle=rng.random() < 0.25)
    elif kind == "batch":
        c.update(n_sims=rng.randint(2, 8), n_min=64, n_max=128, histories=_log(rng, 200_000, 40_000_000))
    elif kind == "learned_dose":
        c.update(photons=_log(rng, 100_000, 40_000_000))
    elif kind == "generate":
        c.update(photons=_log(rng, 500, 10_000_000))
    elif kind == "project":
        c.update(photons=_log(rng, 20_000, 1_500_000), heads=rng.choice([32, 60, 64, 120, 128]),
                 squared=rng.random() < 0.5)
    elif kind == "train":
        c.update(net=rng.choice([GENERATOR, RESPONSE]), batch=_log(rng, 300, 40_000))
    elif kind == "fit_exitplane":
        c.update(photons=_log(rng, 20_000, 300_000), steps=rng.randint(3, 6), batch=_log(rng, 1024, 16384))
    else:
        c.update(photons=_log(rng, 20_000, 300_000), steps=rng.randint(3, 6), batch=_log(rng, 1024, 16384))
    return c


# ---------------------------------------------------------------------- inputs
def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(1_000_003 * int(seed) + salt)


def _uniform(g, lo, hi, n):
    return (lo + (hi - lo) * torch.rand(n, device=DEV, generator=g, dtype=torch.float64)).cpu().numpy()


def _grid(nx, ny, nz, sp):
    ax = [(torch.arange(n, device=DEV, dtype=torch.float32) + 0.5) * sp - n * sp / 2 for n in (nx, ny, nz)]
    return ax[0][None, None, :], ax[1][None, :, None], ax[2][:, None, None]


def _water_labels(nx, ny, nz, seed):
    """uint8 (z, y, x): water with three cortical-bone spheres of 8-15 mm, 2 mm voxels."""
    X, Y, Z = _grid(nx, ny, nz, 2.0)
    lab = torch.zeros(nz, ny, nx, dtype=torch.uint8, device=DEV)
    g = _gen(seed, 1)
    for _ in range(3):
        r = float(_uniform(g, 8.0, 15.0, 1)[0])
        u = _uniform(g, -1.0, 1.0, 3)
        c = [float(u[k] * (n - r)) for k, n in enumerate((nx, ny, nz))]
        lab[(X - c[0]) ** 2 + (Y - c[1]) ** 2 + (Z - c[2]) ** 2 <= r * r] = 1
    return lab.cpu().numpy()


def _ct_hu(nx, ny, nz, seed):
    """int16 HU (z, y, x) on 1 mm voxels: body with noise, two lungs, spine and ribs."""
    g = _gen(seed, 2)
    X, Y, Z = _grid(nx, ny, nz, 1.0)
    X, Y, Z = X * (256.0 / nx), Y * (256.0 / ny), Z * (128.0 / nz)
    hu = torch.full((nz, ny, nx), -1000.0, device=DEV)
    body = (X / 120) ** 2 + (Y / 90) ** 2 + (Z / 62) ** 2 <= 1
    noise = torch.clamp(torch.round(40 + 20 * torch.randn(nz, ny, nx, device=DEV, generator=g)), -50, 110)
    hu = torch.where(body, noise, hu)
    for sx in (-55.0, 55.0):
        lung = ((X - sx) / 35) ** 2 + ((Y - 10) / 45) ** 2 + (Z / 50) ** 2 <= 1
        hu = torch.where(lung & body, torch.full_like(hu, -800.0), hu)
    bone = torch.randint(700, 1201, (nz, ny, nx), device=DEV, generator=g).float()
    spine = ((X / 12) ** 2 + ((Y + 55) / 14) ** 2 <= 1) & body
    ribs = ((torch.sqrt((X / 104) ** 2 + (Y / 78) ** 2) - 1).abs() < 0.035) & (torch.remainder(Z + 200, 24) < 8) \
        & (Y > -60) & body
    hu = torch.where(spine | ribs, bone, hu)
    return hu.to(torch.int16).cpu().numpy()


@functools.lru_cache(maxsize=None)
def _tables(phantom):
    """Physics tables and label rule of a phantom kind (the same for every image)."""
    from opengate_amd import phantoms as P
    from opengate_amd.physics import xs
    from opengate_amd.physics.materials import MaterialDatabase

    db = MaterialDatabase()
    if phantom == "water":
        return xs.build_tables([db.get("G4_WATER"), db.get("G4_BONE_CORTICAL_ICRP")], 0.1406), None, None, None
    if phantom == "batch":
        return xs.build_tables([db.get(n) for n in P.BATCH_MATERIALS], 0.2090), None, None, None
    if phantom == "ct12":
        rows = sorted(P.ct12_materials(db), key=lambda r: r[0])
        mats = [db.get(r[2]) for r in rows] + [db.get("G4_AIR")]
        lut = np.array([0] + list(range(len(rows))) + [0], np.uint16)
        tables = xs.build_tables(mats, 0.1201)
        world = len(mats) - 1
    else:
        import opengate_amd
        from opengate_amd.geometry.materials import HounsfieldUnit_to_material
        from opengate_amd.units import g4_units

        data = Path(opengate_amd.__file__).resolve().parent / "data"
        rows, _ = HounsfieldUnit_to_material(
            SimpleNamespace(volume_manager=SimpleNamespace(material_database=db)), 0.05 * g4_units.g_cm3,
            str(data / "Schneider2000MaterialsTable.txt"), str(data / "Schneider2000DensitiesTable.txt"))
        rows = sorted(rows, key=lambda r: r[0])
        lut = np.array([0] + list(range(1, len(rows) + 1)) + [0], np.uint16)
        used = [0] + [i + 1 for i, r in enumerate(rows) if r[0] < 1250]
        tables = xs.build_tables([db.get("G4_AIR")] + [db.get(r[2]) for r in rows], 0.1201, share_compositions=True,
                                 majorant_materials=np.array(used))
        world = 0
    bins = np.array([r[0] for r in rows] + [rows[-1][1]], np.float64)
    return tables, bins, lut, world


@functools.lru_cache(maxsize=None)
def _spectrum():
    from opengate_amd import phantoms as P

    return P.kramers_spectrum()


def _cone(L):
    """120 kVp point source 600 mm above the phantom centre, 15 deg half-angle cone."""
    from opengate_amd.transport import SourceSpec, spectrum_histogram

    ev, ew, cdf = spectrum_histogram(*_spectrum())
    return SourceSpec(pos_trans=(L[0] / 2, L[1] / 2, L[2] / 2 + 600.0), theta=(0.0, np.deg2rad(15.0)),
                      ene_type="spectrum_histogram", energy_value=ev, energy_width=ew, energy_cdf=cdf)


def _ct_phantom(engine, phantom, nx, ny, nz, seed):
    from opengate_amd.transport import PhantomSpec

    tables, bins, lut, world = _tables(phantom)
    lab = engine.hu_to_labels(_ct_hu(nx, ny, nz, seed), bins, lut)
    L = np.array([nx, ny, nz], float)
    return tables, PhantomSpec(lab.astype(np.uint8), (1.0, 1.0, 1.0), world, tuple(L / 2 - 1500), tuple(L / 2 + 1500))


def _weights(net, seed):
    """FP32 weights (in, out) and biases of a network, padded with zeros to multiples of 8."""
    sizes = [int(s) for s in net.split("-")]
    g = _gen(seed, 3)
    pad = [(s + 7) // 8 * 8 for s in sizes]
    W, b = [], []
    for k, n, pk, pn in zip(sizes[:-1], sizes[1:], pad[:-1], pad[1:]):
        w = torch.zeros(pk, pn, device=DEV)
        w[:k, :n] = torch.randn(k, n, device=DEV, generator=g) * math.sqrt(2.0 / k)
        v = torch.zeros(pn, device=DEV)
        v[:n] = 0.05 * torch.randn(n, device=DEV, generator=g)
        W.append(w)
        b.append(v)
    return sizes, W, b


def _exit_photons(n, seed):
    """Records on the exit plane z = 0 (x y z u v w E weight): aperture of 20 x 20 mm, most
    along the ray from the focal point, a tenth scattered."""
    g = _gen(seed, 4)
    r = lambda: torch.rand(n, device=DEV, generator=g, dtype=torch.float64)  # noqa: E731
    x, y = 22.0 + 20.0 * r(), 22.0 + 20.0 * r()
    d = torch.stack([x - FOCAL[0], y - FOCAL[1], torch.full_like(x, -FOCAL[2])])
    d = d / d.norm(dim=0)
    off = 0.15 * torch.randn(3, n, device=DEV, generator=g, dtype=torch.float64) * (r() < 0.1)
    d = d + off
    d = d / d.norm(dim=0)
    E = 0.02 + 0.1 * (1 - torch.sqrt(r()))
    return [a.float().contiguous() for a in (x, y, torch.zeros_like(x), d[0], d[1], d[2], E, torch.ones_like(x))]


def _frame(nx, ny, nz):
    """Focal frame (e1, e2) of unit vectors n: e1 = (nx nz, ny nz, -up)/up, e2 = (-ny, nx)/up."""
    up = torch.sqrt(nx * nx + ny * ny)
    ok = up > 1e-7
    iu = torch.where(ok, 1 / torch.where(ok, up, torch.ones_like(up)), torch.zeros_like(up))
    zero, one = torch.zeros_like(up), torch.ones_like(up)
    return ((torch.where(ok, nx * nz * iu, nz), torch.where(ok, ny * nz * iu, zero), torch.where(ok, -up, zero)),
            (torch.where(ok, -ny * iu, zero), torch.where(ok, nx * iu, one)))


def _features(rec):
    """(n, 6) FP64 features E, x, y and the direction in the focal frame of the records."""
    x, y, u, v, w, E = (rec[k].double() for k in (0, 1, 3, 4, 5, 6))
    n = torch.stack([x - FOCAL[0], y - FOCAL[1], torch.full_like(x, -FOCAL[2])])
    n = n / n.norm(dim=0)
    (ax, ay, az), (bx, by) = _frame(n[0], n[1], n[2])
    return torch.stack([E, x, y, u * ax + v * ay + w * az, u * bx + v * by, u * n[0] + v * n[1] + w * n[2]], 1)


def _quantiles(F):
    """(6, KNOTS) values of the columns' empirical quantile function at equal Gaussian knots."""
    lev = torch.special.ndtr(torch.linspace(-G_MAX, G_MAX, KNOTS, device=DEV, dtype=torch.float64))
    idx = torch.clamp(torch.round(lev * (F.shape[0] - 1)), 0, F.shape[0] - 1).long()
    return torch.stack([torch.sort(F[:, j]).values[idx] for j in range(F.shape[1])])


def _generator(seed):
    """A generator with seeded weights and quantile tables (as one loaded from a file)."""
    from opengate_amd.learn.exitplane import ExitPlaneGenerator, QuantileMap

    gen = ExitPlaneGenerator(FOCAL, 0.0, device=DEV)
    _, W, b = _weights(GENERATOR, seed)
    gen.mlp.load_state_dict({"W": W, "b": b})
    gen.qmap = QuantileMap(_quantiles(_features(_exit_photons(100_000, seed)).float()), G_MAX)
    return gen


def _escaped(n, L, seed):
    """Photons leaving a cube of side L: on its faces, outward, 140 keV or scattered."""
    g = _gen(seed, 5)
    r = lambda *s: torch.rand(*s, device=DEV, generator=g)  # noqa: E731
    p = r(3, n) * L
    d = torch.randn(3, n, device=DEV, generator=g)
    d = d / d.norm(dim=0)
    face = torch.randint(0, 3, (n,), device=DEV, generator=g)
    i = torch.arange(n, device=DEV)
    p[face, i] = torch.where(d[face, i] > 0, L, 0.0)
    E = torch.where(r(n) < 0.4, torch.full((n,), 0.140511, device=DEV), 0.06 + 0.08 * r(n))
    return [a.contiguous() for a in (*p, *d, E, torch.ones(n, device=DEV))]


def _labelled(n, seed):
    """Rows of the detector-response training set: bf16 (E, theta, phi) scaled, window class."""
    g = _gen(seed, 6)
    X = torch.zeros(n, 8, device=DEV, dtype=torch.bfloat16)
    u = torch.rand(n, 3, device=DEV, generator=g)
    u[:, 1] = u[:, 1] ** 2
    X[:, :3] = (2 * u - 1).to(torch.bfloat16)
    det = torch.rand(n, device=DEV, generator=g) < 0.6 * (1 - u[:, 1])
    cls = torch.where(det, 1 + (u[:, 0] * 2.999).long(), torch.zeros(n, device=DEV, dtype=torch.long))
    return X, cls


HEAD_L = 200.0  # side of the phantom whose photons are projected (mm)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "transport":
        from opengate_amd.transport import GpuEngine, PhantomSpec, SourceSpec, TallySpec

        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        eng = GpuEngine(0)
        if case["phantom"] == "water":
            tables, sp = _tables("water")[0], 2.0
            ph = PhantomSpec(_water_labels(nx, ny, nz, seed), (sp,) * 3)
            src = SourceSpec(pos_trans=(nx * sp / 2, ny * sp / 2, nz * sp / 2), energy=0.1405)
        else:
            sp = 1.0
            tables, ph = _ct_phantom(eng, case["phantom"], nx, ny, nz, seed)
            src = _cone((nx, ny, nz))
        eng.set_physics(tables)
        eng.add_simulation(ph, src, TallySpec(size=(nx, ny, nz), spacing=(sp,) * 3, tle=case["tle"]))
        return {"kind": kind, "eng": eng, "n": [case["histories"]], "seed": 17 + int(seed)}
    if kind == "batch":
        from opengate_amd.transport import GpuEngine, PhantomSpec, SourceSpec, TallySpec, spectrum_lines

        g = _gen(seed, 7)
        eng = GpuEngine(0)
        eng.set_physics(_tables("batch")[0])
        share = _uniform(g, 0.0, math.log(20.0), case["n_sims"])
        share = np.exp(share) / np.exp(share).sum()
        for k in range(case["n_sims"]):
            n = case["n_min"] + k * (case["n_max"] - case["n_min"]) // (case["n_sims"] - 1)
            sp = float(_uniform(g, 1.5, 3.0, 1)[0])
            half = n * sp / 2
            X, Y, Z = _grid(n, n, n, sp)
            a = _uniform(g, 0.6, 0.95, 3) * half
            body = (X / a[0]) ** 2 + (Y / a[1]) ** 2 + (Z / a[2]) ** 2 <= 1
            lab = body.to(torch.uint8)
            for kind_ in (2, 3, 4):  # bone, lung, soft tissue inserts
                e, c = _uniform(g, 0.08, 0.3, 3) * half, _uniform(g, -0.5, 0.5, 3) * a
                ins = ((X - c[0]) / e[0]) ** 2 + ((Y - c[1]) / e[1]) ** 2 + ((Z - c[2]) / e[2]) ** 2 <= 1
                lab[ins & body] = kind_
            s = _uniform(g, 0.2, 0.5, 3) * a
            lines = ([0.140511], [0.885]) if _uniform(g, 0, 1, 1)[0] < 0.5 else ([0.11295, 0.20837], [0.062, 0.104])
            ev, _, cdf = spectrum_lines(*lines)
            src = SourceSpec(pos_type="ellipsoid", pos_param=tuple(s) + (0.0,), pos_trans=(half,) * 3,
                             ene_type="spectrum_discrete", energy_value=ev, energy_cdf=cdf)
            eng.add_simulation(PhantomSpec(lab.cpu().numpy(), (sp,) * 3), src, TallySpec(size=(n,) * 3, spacing=(sp,) * 3))
        return {"kind": kind, "eng": eng, "n": [int(v) for v in share * case["histories"]], "seed": 17 + int(seed)}
    if kind == "learned_dose":
        from opengate_amd.transport import GpuEngine, TallySpec

        n = case["photons"]
        eng = GpuEngine(0)
        tables, ph = _ct_phantom(eng, "ct12", 256, 256, 128, seed)
        eng.set_physics(tables)
        eng.add_simulation(ph, _cone((256, 256, 128)), TallySpec(size=(256, 256, 128)))
        return {"kind": kind, "eng": eng, "gen": _generator(seed), "n": n, "seed": 17 + int(seed),
                "rec": [torch.empty(n, device=DEV) for _ in range(8)]}
    if kind == "generate":
        n = case["photons"]
        return {"kind": kind, "gen": _generator(seed), "n": n, "seed": 17 + int(seed),
                "rec": [torch.empty(n, device=DEV) for _ in range(8)]}
    if kind == "project":
        from opengate_amd.learn.arf import ArfModel, Heads

        arf = ArfModel(device=DEV)
        _, W, b = _weights(RESPONSE, seed)
        arf.mlp.load_state_dict({"W": W, "b": b})
        heads = Heads(center=(HEAD_L / 2,) * 3, radius=HEAD_L / math.sqrt(2.0) + 10.0, n_proj=case["heads"])
        return {"kind": kind, "arf": arf, "heads": heads, "rec": _escaped(case["photons"], HEAD_L, seed),
                "n": case["photons"], "squared": case["squared"]}
    if kind == "train":
        from opengate_amd.learn.mlp import MLP

        sizes, W, b = _weights(case["net"], seed)
        mlp = MLP(sizes, device=DEV)
        mlp.load_state_dict({"W": W, "b": b})
        X, G = _train_batch(case, sizes, seed)
        return {"kind": kind, "mlp": mlp, "X": X, "G": G}
    if kind == "fit_exitplane":
        from opengate_amd.learn.exitplane import ExitPlaneGenerator

        gen = ExitPlaneGenerator(FOCAL, 0.0, device=DEV)
        _, W, b = _weights(GENERATOR, seed)
        gen.mlp.load_state_dict({"W": W, "b": b})
        return {"kind": kind, "gen": gen, "rec": _exit_photons(case["photons"], seed), "steps": case["steps"],
                "batch": case["batch"], "seed": 17 + int(seed)}
    from opengate_amd.learn.arf import ArfModel

    arf = ArfModel(device=DEV)
    _, W, b = _weights(RESPONSE, seed)
    arf.mlp.load_state_dict({"W": W, "b": b})
    X, cls = _labelled(case["photons"], seed)
    return {"kind": kind, "arf": arf, "X": X, "cls": cls, "steps": case["steps"], "batch": case["batch"],
            "seed": 17 + int(seed)}


def _train_batch(case, sizes, seed):
    n = case["batch"]
    g = _gen(seed, 8)
    if sizes[0] == 8:
        X = torch.randn(n, 8, device=DEV, generator=g).to(torch.bfloat16)
    else:
        X = _labelled(n, seed)[0]
    # gradient of a mean loss, with the common part it has before convergence
    return X, (0.5 + torch.randn(n, sizes[-1], device=DEV, generator=g)) / n


# ---------------------------------------------------------------------- one pass
def _dose(eng, n, seed):
    for k in range(len(n)):
        eng.reset_tally(k)
    c = eng.run(n, seed)
    return {"counters": {k: c[k] for k in COUNTERS}, "tally": [eng.get_tally(k) for k in range(len(n))]}


def run(state):
    kind = state["kind"]
    if kind in ("transport", "batch"):
        return _dose(state["eng"], state["n"], state["seed"])
    if kind == "learned_dose":
        from opengate_amd import workloads
        from opengate_amd.transport import SourceSpec

        rec = state["gen"].generate(state["n"], state["seed"], out=state["rec"])
        state["eng"].set_source(0, SourceSpec(pos_type="phsp", phsp=rec, pos_trans=workloads.COLLIMATOR_TO_CT256))
        return _dose(state["eng"], [state["n"]], state["seed"])
    if kind == "generate":
        return state["gen"].generate(state["n"], state["seed"], out=state["rec"])
    if kind == "project":
        from opengate_amd.learn.arf import project

        out = project(state["rec"], state["n"], state["heads"], arf=state["arf"], squared=state["squared"])
        return {k: out[k] for k in ("pairs", "arf", "arf2")}
    if kind == "train":
        mlp = state["mlp"]
        y = mlp.forward(state["X"])
        dW, db = mlp.backward(state["G"])
        mlp.step(dW, db)
        return {"y": y, "dW": dW, "db": db, "W": mlp.W, "b": mlp.b}
    if kind == "fit_exitplane":
        gen = state["gen"]
        loss = gen.fit(state["rec"], steps=state["steps"], batch=state["batch"], seed=state["seed"])
        return {"loss": loss, "qtab": gen.qmap.qtab, "W": gen.mlp.W, "b": gen.mlp.b}
    arf = state["arf"]
    loss = arf.fit(state["X"], state["cls"], steps=state["steps"], batch=state["batch"], seed=state["seed"])
    return {"loss": loss, "W": arf.mlp.W, "b": arf.mlp.b}


# ---------------------------------------------------------------------- work
def _madds(net):
    s = [int(v) for v in net.split("-")]
    return sum(k * n for k, n in zip(s[:-1], s[1:])), sum(k * n for k, n in zip(s[1:-1], s[2:]))


def work(case):
    kind = case["kind"]
    if kind in ("transport", "batch", "learned_dose"):
        # a history: about 13 tentative steps (a logarithm, a move, a label, an interpolation),
        # its birth and its interactions: some 1000 FP32 operations; labels read once, two FP64
        # tally images written once
        n = case["photons"] if kind == "learned_dose" else case["histories"]
        vox = {"transport": lambda: case["nx"] * case["ny"] * case["nz"], "learned_dose": lambda: 256 * 256 * 128,
               "batch": lambda: case["n_sims"] * 96 ** 3}[kind]()
        flops = 1000.0 * n
        if kind == "learned_dose":
            flops += 2.0 * _madds(GENERATOR)[0] * n
        return {"bytes": 17.0 * vox, "flops": flops}
    if kind == "generate":
        return {"bytes": 32.0 * case["photons"], "flops": 2.0 * _madds(GENERATOR)[0] * case["photons"]}
    if kind == "project":
        # about 0.05 pairs a photon and head at 128 heads; images of 128 x 128 pixels, 3 windows
        pairs = case["photons"] * 0.0075 * case["heads"]
        img = case["heads"] * 3 * 128 * 128 * 8.0 * (2 if case["squared"] else 1)
        return {"bytes": 32.0 * case["photons"] + img, "flops": 2.0 * _madds(RESPONSE)[0] * pairs}
    net, steps, n = {"train": lambda: (case["net"], 1, case["batch"]),
                     "fit_exitplane": lambda: (GENERATOR, case["steps"], case["batch"]),
                     "fit_response": lambda: (RESPONSE, case["steps"], case["batch"])}[kind]()
    full, inner = _madds(net)
    s = [int(v) for v in net.split("-")]
    # Adam: parameter and two moments read and written; batch read, output and its gradient
    rows = {"train": 0, "fit_exitplane": 32.0 * case.get("photons", 0), "fit_response": 24.0 * case.get("photons", 0)}
    return {"bytes": steps * (24.0 * full + n * (2.0 * s[0] + 8.0 * s[-1])) + rows[kind],
            "flops": steps * n * 2.0 * (2 * full + inner)}


# ---------------------------------------------------------------------- exact values
def _forward64(sizes, W, b, x):
    """Layer inputs and pre-activations of the network in FP64 (unpadded weights)."""
    xs, zs = [x], []
    for i, (k, n) in enumerate(zip(sizes[:-1], sizes[1:])):
        zs.append(xs[-1] @ W[i][:k, :n] + b[i][:n])
        if i < len(sizes) - 2:
            xs.append(torch.relu(zs[-1]))
    return xs, zs


def _philox(c0, c1, c2, c3, k0, k1):
    """Philox4x32-10 (Salmon et al., SC11) on int64 tensors of 32-bit words."""
    m32 = 0xFFFFFFFF

    def mul(a, x):
        lo16, hi16 = x & 0xFFFF, x >> 16
        low = a * lo16
        mid = a * hi16 + (low >> 16)
        return (mid >> 16) & m32, ((mid & 0xFFFF) << 16) | (low & 0xFFFF)

    for _ in range(10):
        h0, l0 = mul(0xD2511F53, c0)
        h1, l1 = mul(0xCD9E8D57, c2)
        c0, c1, c2, c3 = h1 ^ c1 ^ k0, l1, h0 ^ c3 ^ k1, l0
        k0, k1 = (k0 + 0x9E3779B9) & m32, (k1 + 0xBB67AE85) & m32
    return c0, c1, c2, c3


def _noise64(n, seed, first, cols=8):
    """The generator's N(0,1) noise, rows first..first+n-1, rounded to bf16 (its input format)."""
    row = first + torch.arange(n, device=DEV, dtype=torch.int64)
    out = torch.empty(n, cols, device=DEV, dtype=torch.float64)
    for blk in range(cols // 4):
        w = _philox(row & 0xFFFFFFFF, row >> 32, torch.full_like(row, 0x4E4F4953), torch.full_like(row, blk),
                    seed & 0xFFFFFFFF, seed >> 32)
        u = [((x >> 8) | 1).double() * 2.0 ** -24 for x in w]
        for j in (0, 2):
            r, a = torch.sqrt(-2 * torch.log(u[j])), 2 * math.pi * u[j + 1]
            out[:, 4 * blk + j], out[:, 4 * blk + j + 1] = r * torch.cos(a), r * torch.sin(a)
    return out.float().to(torch.bfloat16).double()


def _decode64(Z, q):
    t = torch.clamp((Z + G_MAX) * ((KNOTS - 1) / (2 * G_MAX)), 0, KNOTS - 1)
    k = torch.clamp(t.long(), max=KNOTS - 2)
    a = t - k
    E, px, py, lu, lv, lw = (q[j][k[:, j]] + a[:, j] * (q[j][k[:, j] + 1] - q[j][k[:, j]]) for j in range(6))
    d = torch.stack([lu, lv, lw])
    d = d / d.norm(dim=0)
    m = torch.stack([px - FOCAL[0], py - FOCAL[1], torch.full_like(px, -FOCAL[2])])
    m = m / m.norm(dim=0)
    (ax, ay, az), (bx, by) = _frame(m[0], m[1], m[2])
    o = torch.stack([d[2] * m[0] + d[1] * bx + d[0] * ax, d[2] * m[1] + d[1] * by + d[0] * ay, d[2] * m[2] + d[0] * az])
    o = o / o.norm(dim=0)
    return [px, py, torch.zeros_like(px), o[0], o[1], o[2], E, torch.ones_like(px)]


def _bf16_weights64(net, seed):
    sizes, W, b = _weights(net, seed)
    return sizes, [w.to(torch.bfloat16).double() for w in W], [v.double() for v in b]


def _adam64(p, g, m, v, t, lr):
    m.mul_(0.9).add_(g, alpha=0.1)
    v.mul_(0.999).addcmul_(g, g, value=0.001)
    p.sub_(lr * (m / (1 - 0.9 ** t)) / (torch.sqrt(v / (1 - 0.999 ** t)) + 1e-8))


def _pad64(t, like):
    out = torch.zeros(like.shape, device=DEV, dtype=torch.float64)
    out[tuple(slice(0, s) for s in t.shape)] = t
    return out


def _fit64(net, seed, steps, lr, lr_min, batches):
    """Losses and weights of `steps` Adam steps in FP64; batches(it) -> (x, loss(output))."""
    sizes, Wp, bp = _weights(net, seed)
    P = [w[:k, :n].double().clone() for w, k, n in zip(Wp, sizes[:-1], sizes[1:])]
    P += [v[:n].double().clone() for v, n in zip(bp, sizes[1:])]
    M, V, L = [torch.zeros_like(p) for p in P], [torch.zeros_like(p) for p in P], len(sizes) - 1
    losses = []
    for it in range(steps):
        x, loss = batches(it)
        Q = [p.clone().requires_grad_(True) for p in P]
        h = x
        for i in range(L):
            h = h @ Q[i] + Q[L + i]
            if i < L - 1:
                h = torch.relu(h)
        val = loss(h)
        val.backward()
        losses.append(float(val.detach()))
        rate = lr_min + 0.5 * (lr - lr_min) * (1 + math.cos(math.pi * it / max(1, steps)))
        for p, q, m, v in zip(P, Q, M, V):
            _adam64(p, q.grad, m, v, it + 1, rate)
    return np.array(losses), [_pad64(p, w) for p, w in zip(P[:L], Wp)]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("transport", "batch", "learned_dose"):
        return None  # follows the framework's own random streams
    if kind == "generate":
        sizes, W, b = _bf16_weights64(GENERATOR, seed)
        q = _quantiles(_features(_exit_photons(100_000, seed)).float()).double()
        parts = []
        for s in range(0, case["photons"], 1 << 20):
            n = min(1 << 20, case["photons"] - s)
            Z = _forward64(sizes, W, b, _noise64(n, 17 + int(seed), s))[1][-1]
            parts.append(_decode64(Z, q))
        return [torch.cat(a) for a in zip(*parts)]
    if kind == "project":
        return _project64(case, seed)
    if kind == "train":
        sizes, W, b = _bf16_weights64(case["net"], seed)
        X, G = _train_batch(case, sizes, seed)
        xs, zs = _forward64(sizes, W, b, X[:, :sizes[0]].double())
        _, Wp, bp = _weights(case["net"], seed)
        g, dW, db, Wn = G.double(), [], [], []
        for i in range(len(W) - 1, -1, -1):
            dW.insert(0, xs[i].T @ g)
            db.insert(0, g.sum(0))
            if i:
                g = (g @ W[i][:sizes[i], :sizes[i + 1]].T) * (zs[i - 1] > 0)
        for w, d in zip(Wp, dW):
            p = w[:d.shape[0], :d.shape[1]].double().clone()
            _adam64(p, d, torch.zeros_like(p), torch.zeros_like(p), 1, 1e-3)
            Wn.append(_pad64(p, w))
        # (a bias after one Adam step is its start plus or minus the rate: no value to compare)
        return {"y": zs[-1], "dW": [_pad64(d, w) for d, w in zip(dW, Wp)], "db": [_pad64(d, v) for d, v in zip(db, bp)],
                "W": Wn, "b": None}
    if kind == "fit_exitplane":
        F = _features(_exit_photons(case["photons"], seed)).float().double()
        N, s = F.shape[0], 17 + int(seed)
        ar = (torch.arange(N, device=DEV, dtype=torch.float64) + 0.5) / N
        T = torch.empty_like(F)
        for j in range(6):
            T[torch.argsort(F[:, j], stable=True), j] = torch.special.ndtri(ar)
        g, batch = torch.Generator(device=DEV).manual_seed(s), case["batch"]

        def batches(it):
            d = T[torch.randint(0, N, (batch,), device=DEV, generator=g)]
            th = torch.randn(6, 128, device=DEV, generator=g).double()
            th = torch.cat([th / th.norm(dim=0, keepdim=True), torch.eye(6, device=DEV, dtype=torch.float64)], 1)
            return _noise64(batch, s * 1_000_003 + 17, it * batch), lambda o: (
                (torch.sort(o @ th, 0).values - torch.sort(d @ th, 0).values) ** 2).mean()

        loss, W = _fit64(GENERATOR, seed, case["steps"], 1e-3, 3e-5, batches)
        return {"loss": loss, "qtab": _quantiles(F), "W": W, "b": None}
    X, cls = _labelled(case["photons"], seed)
    g = torch.Generator(device=DEV).manual_seed(17 + int(seed))

    def batches(it):
        i = torch.randint(0, X.shape[0], (case["batch"],), device=DEV, generator=g)
        return X[i, :3].double(), lambda z: torch.nn.functional.cross_entropy(z, cls[i])

    loss, W = _fit64(RESPONSE, seed, case["steps"], 2e-3, 5e-5, batches)
    return {"loss": loss, "W": W, "b": None}


def _project64(case, seed):
    """Window probabilities of every (photon, head) pair added into the projection images."""
    H, sizes = case["heads"], [int(s) for s in RESPONSE.split("-")]
    _, W, b = _bf16_weights64(RESPONSE, seed)
    rec = [a.double() for a in _escaped(case["photons"], HEAD_L, seed)]
    # axis to face; face to mid-crystal (35 mm of holes, 1 mm gap, half of 9.5 mm); acceptance; pixel
    radius, depth, tmax, sp = HEAD_L / math.sqrt(2.0) + 10.0, 40.75, math.radians(10.0), 4.8
    lo, hi = 0.010, 0.160  # energies scaled to [-1, 1], MeV
    img = torch.zeros(H, 3, 128 * 128, device=DEV, dtype=torch.float64)
    img2, pairs = torch.zeros_like(img), 0
    x, y, z = (rec[k] - HEAD_L / 2 for k in range(3))
    u, v, w, E, wt = rec[3:]
    for k in range(H):
        ca, sa = math.cos(2 * math.pi * k / H), math.sin(2 * math.pi * k / H)
        c = u * ca + v * sa
        t = (radius - (x * ca + y * sa)) / c
        i = torch.nonzero((c > math.cos(tmax)) & (t >= 0))[:, 0]
        c, t = c[i], t[i]
        dy = -u[i] * sa + v[i] * ca
        hu = -(x[i] + t * u[i]) * sa + (y[i] + t * v[i]) * ca + depth / c * dy
        hz = z[i] + t * w[i] + depth / c * w[i]
        ix, iy = torch.floor((hu + 64 * sp) / sp).long(), torch.floor((hz + 64 * sp) / sp).long()
        ok = (ix >= 0) & (iy >= 0) & (ix < 128) & (iy < 128)
        X = torch.stack([E[i] * (2 / (hi - lo)) - (hi + lo) / (hi - lo),
                         torch.acos(torch.clamp(c, max=1.0)) * (2 / tmax) - 1, torch.atan2(dy, w[i]) / math.pi], 1)[ok]
        p = torch.softmax(_forward64(sizes, W, b, X)[1][-1], 1)[:, 1:] * wt[i][ok][:, None]
        pix = (iy * 128 + ix)[ok]
        for a in range(3):
            img[k, a].index_add_(0, pix, p[:, a])
            img2[k, a].index_add_(0, pix, p[:, a] ** 2)
        pairs += int(ok.sum())
    out = {"pairs": None, "arf": img.view(H * 3, 128, 128)}
    out["arf2"] = img2.view(H * 3, 128, 128) if case["squared"] else None
    return out
