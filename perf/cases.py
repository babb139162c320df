"""The work that a user's program has this framework do, as measurable cases.

Every case goes through the package's public entry points: time steps of one
ferromagnet (World, Ferromagnet, TimeSolver), of an antiferromagnet with
elastodynamics, of many small magnets together (Batch), the quantities that an
output table is made of, and the demag operator on the caller's own device
arrays.  `exact` restates the same physics in 64 bits with plain torch.
"""

import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "mumax-plus_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

MU0, GAMMA = 1.25663706212e-6, 1.7595e11
QE, MUB = 1.60217646e-19, 9.274009152e-24
DEV = "cuda"

# Case fields (kind "llg", one ferromagnet): size; cell in-plane cell size (m)
# and cz its height; steps fixed steps of dt with `method`, or, with
# `duration` > 0, an adaptive run of that simulated time; dmi interfacial DMI
# (J/m2), ku uniaxial anisotropy (J/m3) along z, bias a field (T) along x;
# disk: elliptical geometry mask; grains: msat and ku vary from grain to
# grain (per-cell parameters); pbc: image repetitions along x and y; jcur a
# current density along x (Zhang-Li torque); m0 "random" or "smooth".
_LLG = {"kind": "llg", "nx": 0, "ny": 0, "nz": 1, "cell": 4e-9, "cz": 4e-9, "method": "DormandPrince", "steps": 0,
        "dt": 5e-14, "duration": 0.0, "msat": 8e5, "aex": 1.3e-11, "alpha": 0.02, "dmi": 0.0, "ku": 0.0, "bias": 0.0,
        "disk": False, "grains": False, "pbc": 0, "jcur": 0.0, "m0": "smooth"}


def _llg(**kw):
    return {**_LLG, **kw}


def listed():
    return [
        # the smallest solves: an elliptical nanodisk, a hundred launches a step
        _llg(name="disk_40x24", nx=40, ny=24, cell=2e-9, cz=2e-9, steps=20, dt=1e-13, msat=1e6, ku=4e5, alpha=0.05,
             bias=0.05, disk=True),
        # the thin film of the introductory scripts: adaptive run in a field
        _llg(name="film_128x32_adaptive", nx=128, ny=32, cell=3.906e-9, cz=3e-9, duration=1e-11, bias=0.025),
        # a granular few-layer medium: per-cell parameters, ragged sizes, the default method, a mask
        _llg(name="grains_190x150x3", nx=190, ny=150, nz=3, method="Fehlberg", steps=10, msat=6e5, ku=3e5, disk=True,
             grains=True),
        # a current-driven texture in a racetrack: Zhang-Li torque and DMI
        _llg(name="track_500x100_stt", nx=500, ny=100, cell=2e-9, cz=1e-9, steps=10, msat=5.8e5, aex=1.5e-11, alpha=0.3,
             dmi=3e-3, ku=8e5, jcur=1e12),
        # a large skyrmion film
        _llg(name="film_1024x1024_dmi", nx=1024, ny=1024, cell=2e-9, cz=1e-9, steps=10, msat=5.8e5, aex=1.5e-11,
             alpha=0.1, dmi=3e-3, ku=8e5, bias=0.01),
        # a multilayer of ragged size with uniform parameters
        _llg(name="layers_300x220x6", nx=300, ny=220, nz=6, cell=3e-9, cz=2e-9, steps=10, ku=2e5, dmi=1e-3),
        # the benchmark's block
        _llg(name="bulk_256x256x64", nx=256, ny=256, nz=64, cell=2e-9, cz=2e-9, steps=10, msat=1.1e6, aex=1.6e-11,
             alpha=0.0, dmi=3e-3, ku=8e5, m0="random"),
        # the benchmark's antiferromagnet with magnetoelastic coupling and elastodynamics
        {"name": "afm_512x512_elastic", "kind": "afm", "nx": 512, "ny": 512, "steps": 10, "elastic": True},
        # the benchmark's batch of small magnets, a short solve of each
        {"name": "batch_256", "kind": "batch", "members": 256, "steps": 40, "lo": 4.0, "hi": 7.0, "layers": 2.0,
         "pow2": True},
        # one row of an output table with its fields
        {"name": "table_240x130x2", "kind": "table", "nx": 240, "ny": 130, "nz": 2},
        # the operator on device arrays, thick and ragged
        {"name": "demag_200x120x40", "kind": "demag", "nx": 200, "ny": 120, "nz": 40, "pbc": 0, "geom": True},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("film", "film", "layers", "bulk", "track", "afm", "batch", "table", "demag"))
    if kind == "film":
        nx, ny = _logint(rng, 20, 1024), _logint(rng, 16, 1024)
        dmi = rng.choice((0.0, 1e-3, 3e-3))
        return _llg(nx=nx, ny=ny, cell=2e-9, cz=rng.choice((1e-9, 3e-9)), steps=rng.choice((5, 10, 20)), dmi=dmi,
                    ku=rng.choice((0.0, 5e5)), bias=rng.choice((0.0, 0.02)), disk=rng.random() < 0.3,
                    grains=rng.random() < 0.25, pbc=rng.choice((0, 0, 2)),
                    method=rng.choice(("DormandPrince", "Fehlberg", "BogackiShampine", "Heun")))
    if kind == "layers":
        return _llg(nx=_logint(rng, 20, 400), ny=_logint(rng, 20, 400), nz=rng.randint(2, 9), cell=3e-9, cz=2e-9,
                    steps=rng.choice((5, 10)), ku=2e5, dmi=rng.choice((0.0, 1e-3)), disk=rng.random() < 0.3,
                    grains=rng.random() < 0.3, method=rng.choice(("DormandPrince", "Fehlberg")))
    if kind == "bulk":
        return _llg(nx=_logint(rng, 40, 256), ny=_logint(rng, 40, 256), nz=rng.randint(10, 64), cell=2e-9, cz=2e-9,
                    steps=rng.choice((4, 8)), msat=1.1e6, aex=1.6e-11, alpha=rng.choice((0.0, 0.1)),
                    dmi=rng.choice((0.0, 3e-3)), ku=8e5)
    if kind == "track":
        return _llg(nx=_logint(rng, 100, 1000), ny=_logint(rng, 20, 200), cell=2e-9, cz=1e-9, steps=10, msat=5.8e5,
                    aex=1.5e-11, alpha=0.3, dmi=3e-3, ku=8e5, jcur=rng.uniform(5e11, 2e12))
    if kind == "afm":
        return {"kind": "afm", "nx": _logint(rng, 48, 512), "ny": _logint(rng, 48, 512), "steps": 10,
                "elastic": rng.random() < 0.6}
    if kind == "batch":
        return {"kind": "batch", "members": _logint(rng, 8, 200), "steps": rng.choice((10, 20)), "lo": 3.5,
                "hi": rng.uniform(5.0, 6.8), "layers": rng.choice((0.0, 1.6, 2.0)), "pow2": rng.random() < 0.3}
    if kind == "table":
        return {"kind": "table", "nx": _logint(rng, 30, 500), "ny": _logint(rng, 30, 300), "nz": rng.randint(1, 4)}
    return {"kind": "demag", "nx": _logint(rng, 24, 300), "ny": _logint(rng, 24, 300), "nz": _logint(rng, 1, 48),
            "pbc": rng.choice((0, 0, 1)), "geom": rng.random() < 0.5}


# ------------------------------------------------------------------ inputs

def _smooth(rng, shape, mean=(0.0, 0.0, 0.0), noise=0.05):
    """Unit vectors from a few long waves and a little noise: a texture as
    relaxations and switching runs meet it."""
    nz, ny, nx = shape
    z, y, x = np.meshgrid(*(np.arange(n) / max(n, 8) for n in shape), indexing="ij", sparse=True)
    m = rng.normal(size=(3,) + shape) * noise
    for c in range(3):
        m[c] += mean[c]
        for _ in range(3):
            kx, ky, kz = rng.integers(-2, 3, 3)
            m[c] += rng.normal() * np.cos(2 * np.pi * (kx * x + ky * y + kz * z) + rng.uniform(0, 2 * np.pi))
    return (m / np.linalg.norm(m, axis=0)).astype(np.float32)


def _random(rng, shape):
    m = rng.normal(size=(3,) + shape)
    return (m / np.linalg.norm(m, axis=0)).astype(np.float32)


def _disk(shape):
    nz, ny, nx = shape
    x, y = (np.arange(nx) - (nx - 1) / 2) / (nx / 2), (np.arange(ny) - (ny - 1) / 2) / (ny / 2)
    return np.broadcast_to((x[None, :] ** 2 + y[:, None] ** 2 <= 1.0), shape).copy()


def _grains(rng, shape, size=12):
    """Per-cell factors, one per grain of a square grain pattern with ragged edges."""
    nz, ny, nx = shape
    jx, jy = rng.integers(0, 3, (ny, nx)), rng.integers(0, 3, (ny, nx))
    gx, gy = (np.arange(nx)[None, :] + jx) // size, (np.arange(ny)[:, None] + jy) // size
    f = rng.uniform(0.8, 1.2, (ny // size + 2, nx // size + 2))
    return np.broadcast_to(f[gy, gx], shape).astype(np.float32).copy()


def _llg_inputs(case, seed):
    rng = np.random.default_rng(seed)
    shape = (case["nz"], case["ny"], case["nx"])
    m0 = _random(rng, shape) if case["m0"] == "random" else _smooth(rng, shape)
    geom = _disk(shape) if case["disk"] else None
    msat, ku = case["msat"], case["ku"]
    if case["grains"]:
        f = _grains(rng, shape)
        msat, ku = (msat * f).astype(np.float32), (ku * f[:, ::-1]).astype(np.float32)
    return m0, geom, msat, ku


_BATCH_P = (("msat", 4e5, 1.4e6), ("aex", 5e-12, 2e-11), ("ku1", 0.0, 1e6), ("alpha", 0.005, 0.1))
_BATCH_DT = 2e-14  # within the stability limit of the stiffest draw (A 2e-11 J/m, Ms 4e5 A/m, 2 nm cells)


def _batch_inputs(case, seed):
    # the sizes belong to the case, the states and materials to the seed
    sizes, rng = np.random.default_rng(case["members"]), np.random.default_rng(seed)
    rnd = (lambda v: int(2 ** round(v))) if case["pow2"] else (lambda v: int(round(2 ** v)))
    out = []
    for _ in range(case["members"]):
        nx, ny = (rnd(v) for v in sizes.uniform(case["lo"], case["hi"], 2))
        nz = rnd(sizes.uniform(0, case["layers"]))
        p = {k: float(np.float32(rng.uniform(lo, hi))) for k, lo, hi in _BATCH_P}
        out.append(((nx, ny, nz), p, _smooth(rng, (nz, ny, nx))))
    return out


# Antiferromagnet of the benchmark (2 nm cells, periodic in x and y).
_AFM = {"msat": 566e3, "aex": 2.48e-12, "alpha": 0.004, "afmex_cell": -4e-12, "dmi": 1e-3, "B": -8.8e6, "C11": 283e9,
        "C12": 166e9, "C44": 58e9, "rho": 8900.0, "eta": 1e10, "latcon": 0.35e-9, "dt": 1e-14, "reps": 2}


def _afm_inputs(case, seed):
    rng = np.random.default_rng(seed)
    shape = (1, case["ny"], case["nx"])
    m1 = _random(rng, shape)
    m2 = (-m1 + 0.01 * rng.normal(size=m1.shape)).astype(np.float32)
    # a displacement as a run in progress has it, so that the elastic state counts from the first step
    u = np.zeros((3,) + shape, dtype=np.float32)
    y, x = np.arange(case["ny"])[:, None] / case["ny"], np.arange(case["nx"])[None, :] / case["nx"]
    for c in range(3):
        for _ in range(3):
            kx, ky = rng.integers(-3, 4, 2)
            u[c, 0] += 1e-13 * rng.normal() * np.sin(2 * np.pi * (kx * x + ky * y) + rng.uniform(0, 6.28))
    return m1, m2, u


# ------------------------------------------------------------------ prepare / run

def prepare(case, seed):
    import mumaxplus as mp
    kind = case["kind"]
    if kind == "llg" or kind == "table":
        if kind == "table":
            case = _llg(nx=case["nx"], ny=case["ny"], nz=case["nz"], steps=2, dt=1e-13, alpha=0.1, bias=0.02, ku=1e5)
        m0, geom, msat, ku = _llg_inputs(case, seed)
        size = (case["nx"], case["ny"], case["nz"])
        reps = case["pbc"]
        pbc = {"mastergrid": mp.Grid((size[0], size[1], 0)), "pbc_repetitions": (reps, reps, 0)} if reps else {}
        world = mp.World((case["cell"], case["cell"], case["cz"]), **pbc)
        mag = mp.Ferromagnet(world, mp.Grid(size), geometry=geom)
        mag.msat, mag.aex, mag.alpha = msat, case["aex"], case["alpha"]
        if case["ku"]:
            mag.ku1, mag.anisU = ku, (0, 0, 1)
        if case["dmi"]:
            mag.dmi_tensor.set_interfacial_dmi(case["dmi"])
        if case["bias"]:
            mag.bias_magnetic_field = (case["bias"], 0, 0)
        if case["jcur"]:
            mag.jcur, mag.xi, mag.pol = (case["jcur"], 0, 0), 0.2, 0.6
        mag.magnetization = m0
        ts = world.timesolver
        ts.set_method(case["method"])
        if case["duration"]:
            ts.adaptive_timestep = True
        else:
            ts.adaptive_timestep, ts.timestep = False, case["dt"]
        return {"case": case, "kind": kind, "world": world, "mag": mag, "m0": m0}
    if kind == "afm":
        m1, m2, u = _afm_inputs(case, seed)
        nx, ny, c, p = case["nx"], case["ny"], 2e-9, _AFM
        world = mp.World((c, c, c), mastergrid=mp.Grid((nx, ny, 0)), pbc_repetitions=(p["reps"], p["reps"], 0))
        afm = mp.Antiferromagnet(world, mp.Grid((nx, ny, 1)))
        afm.msat, afm.aex, afm.alpha, afm.afmex_cell = p["msat"], p["aex"], p["alpha"], p["afmex_cell"]
        afm.dmi_tensors.set_bulk_dmi(p["dmi"])
        if case["elastic"]:
            afm.B1 = afm.B2 = p["B"]
            afm.enable_elastodynamics = True
            afm.C11, afm.C12, afm.C44, afm.rho, afm.eta = p["C11"], p["C12"], p["C44"], p["rho"], p["eta"]
            afm.elastic_displacement = u
        afm.sub1.magnetization, afm.sub2.magnetization = m1, m2
        ts = world.timesolver
        ts.set_method("DormandPrince")
        ts.adaptive_timestep, ts.timestep = False, p["dt"]
        return {"case": case, "kind": kind, "world": world, "afm": afm}
    if kind == "batch":
        mags, span = [], 0
        for (nx, ny, nz), p, m0 in _batch_inputs(case, seed):
            world = mp.World((2e-9, 2e-9, 2e-9))
            mag = mp.Ferromagnet(world, mp.Grid((nx, ny, nz)))
            mag.msat, mag.aex, mag.ku1, mag.anisU, mag.alpha = p["msat"], p["aex"], p["ku1"], (0, 0, 1), p["alpha"]
            mag.magnetization = m0
            ts = world.timesolver
            ts.set_method("DormandPrince")
            ts.adaptive_timestep, ts.timestep = False, _BATCH_DT
            mags.append(mag)
            span += -(-nx * ny * nz // 256) * 256
        return {"case": case, "kind": kind, "mags": mags, "batch": mp.Batch(span)}
    # demag: the caller's own arrays; a program keeps its plan
    g = torch.Generator(device=DEV).manual_seed(seed)
    shape = (case["nz"], case["ny"], case["nx"])
    m = torch.randn((3,) + shape, generator=g, device=DEV)
    m /= m.norm(dim=0)
    geom = torch.from_numpy(_disk(shape).astype(np.uint8)).to(DEV) if case["geom"] else None
    box, reps = ((case["nx"], case["ny"], 0), (case["pbc"],) * 2 + (0,)) if case["pbc"] else ((0, 0, 0), (0, 0, 0))
    plan = mp._cpp.DemagPlan((case["nx"], case["ny"], case["nz"]), (4e-9, 4e-9, 4e-9), box, reps)
    return {"case": case, "kind": kind, "plan": plan, "m": m, "geom": geom, "h": torch.empty_like(m)}


def run(state):
    kind, case = state["kind"], state["case"]
    if kind == "llg":
        ts = state["world"].timesolver
        if case["duration"]:
            # a leg of a sweep: the state is set, run and read
            state["mag"].magnetization = state["m0"]
            ts.run(case["duration"])
        else:
            ts.steps(case["steps"])
        return state["mag"].magnetization.get()
    if kind == "table":
        mag = state["mag"]
        state["world"].timesolver.steps(case["steps"])
        return {"average": np.array(mag.magnetization.average()), "energy": mag.total_energy(),
                "torque": mag.max_torque(), "demag": mag.demag_field(), "field": mag.effective_field(),
                "m": mag.magnetization.get()}
    if kind == "afm":
        state["world"].timesolver.steps(case["steps"])
        a = state["afm"]
        out = [a.sub1.magnetization.get(), a.sub2.magnetization.get()]
        if case["elastic"]:
            out += [a.elastic_displacement.get(), a.elastic_velocity.get()]
        return out
    if kind == "batch":
        batch = state["batch"]
        for mag in state["mags"]:
            batch.add(mag, steps=case["steps"])
        batch.run_until_done(poll=case["steps"])
        got = [mag.magnetization.get().reshape(-1) for mag in state["mags"]]
        per = -(-len(got) // 32)
        return [np.concatenate(got[i:i + per]) for i in range(0, len(got), per)]
    geom = state["geom"]
    state["plan"].exec(state["m"].data_ptr(), state["h"].data_ptr(), 8e5, None, None if geom is None else geom.data_ptr(),
                       torch.cuda.current_stream().cuda_stream)
    return state["h"]


# ------------------------------------------------------------------ work, tolerance

def _field_work(nx, ny, nz, sources=1):
    """Bytes and flops of one field evaluation: the state read, its field
    written and the real spectrum of the kernel read once; three forward and
    three inverse real transforms of the grid padded to twice its size, the
    tensor product, and about 150 operations a cell for the local terms."""
    n = nx * ny * nz
    p = math.prod(2 * k if k > 1 else 1 for k in (nx, ny, nz))
    octant = math.prod(k + 1 if k > 1 else 1 for k in (nx, ny, nz))
    return 24.0 * n * sources + 24.0 * octant, 6 * 2.5 * p * math.log2(p) + 15.0 * p + 150.0 * n * sources


_EVALS = {"DormandPrince": 6, "Fehlberg": 6, "BogackiShampine": 3, "Heun": 2}


def work(case):
    kind = case["kind"]
    if kind == "batch":
        got = [_field_work(*size) for size, _, _ in _batch_inputs(case, 0)]
        e = 6 * case["steps"]
        return {"bytes": e * sum(b for b, _ in got), "flops": e * sum(f for _, f in got)}
    nx, ny, nz = case["nx"], case["ny"], case.get("nz", 1)
    b, f = _field_work(nx, ny, nz, 2 if kind == "afm" else 1)
    if kind == "llg":
        # an adaptive run takes steps of some 3e-13 s
        e = _EVALS[case["method"]] * (case["steps"] or math.ceil(case["duration"] / 3e-13))
    elif kind == "afm":
        e = 6 * case["steps"]
        if case["elastic"]:
            b, f = b + 48.0 * nx * ny, f + 200.0 * nx * ny
    elif kind == "table":
        e = 6 * 2 + 4
    else:
        e = 1
    return {"bytes": e * b, "flops": e * f}


def tolerance(case):
    # about four times the distance from `exact` that was measured: 2e-7 to
    # 3e-7 for a field, 1e-7 to 3.4e-6 after time steps, where the differences
    # of single cells grow (most where neighbours point at random, or where
    # the step controller takes other steps since an error norm rounds otherwise)
    if case["kind"] in ("demag", "table"):
        return {"rel": 1e-6, "max": 1e-4}
    return {"rel": 1.4e-5, "max": 3e-3}


# ------------------------------------------------------------------ the same in 64 bits

def _newell(n, cell, box=(0, 0, 0), reps=(0, 0, 0)):
    """The demag tensor (xx, yy, zz, xy, xz, yz) on the offsets 0..n-1 with
    its images: second differences of Newell's f and g (J. Geophys. Res. 98,
    9551 (1993), eqs. 27 and 32)."""
    def axis(k, shift):
        return torch.arange(-1, n[k] + 1, dtype=torch.float64, device=DEV) * cell[k] + shift * cell[k]

    def xlog(w, a, b):  # w asinh(a / b), zero where b is
        return torch.where(b > 0, w * torch.asinh(a / torch.where(b > 0, b, 1.0)), 0.0)

    def xatan(w, a, b):
        return torch.where(b != 0, w * torch.atan(a / torch.where(b != 0, b, 1.0)), 0.0)

    def f(x, y, z):
        r = torch.sqrt(x * x + y * y + z * z)
        return (xlog(0.5 * y * (z * z - x * x), y, torch.sqrt(x * x + z * z)) +
                xlog(0.5 * z * (y * y - x * x), z, torch.sqrt(x * x + y * y)) -
                xatan(x * y * z, y * z, x * r) + (2 * x * x - y * y - z * z) * r / 6)

    def g(x, y, z):
        r = torch.sqrt(x * x + y * y + z * z)
        return (xlog(x * y * z, z, torch.sqrt(x * x + y * y)) +
                xlog(y * (3 * z * z - y * y) / 6, x, torch.sqrt(y * y + z * z)) +
                xlog(x * (3 * z * z - x * x) / 6, y, torch.sqrt(x * x + z * z)) -
                xatan(z ** 3 / 6, x * y, z * r) - xatan(z * y * y / 2, x * z, y * r) -
                xatan(z * x * x / 2, y * z, x * r) - x * y * r / 3)

    def diff(v):
        for d in (0, 1, 2):
            k = v.shape[d]
            v = 2 * v.narrow(d, 1, k - 2) - v.narrow(d, 0, k - 2) - v.narrow(d, 2, k - 2)
        return v / (4 * math.pi * cell[0] * cell[1] * cell[2])

    out = torch.zeros((6, n[2], n[1], n[0]), dtype=torch.float64, device=DEV)
    for i in range(-reps[0], reps[0] + 1):
        for j in range(-reps[1], reps[1] + 1):
            for k in range(-reps[2], reps[2] + 1):
                x = axis(0, i * box[0])[None, None, :]
                y = axis(1, j * box[1])[None, :, None]
                z = axis(2, k * box[2])[:, None, None]
                for c, (fn, a) in enumerate(((f, (x, y, z)), (f, (y, z, x)), (f, (z, x, y)), (g, (x, y, z)),
                                             (g, (x, z, y)), (g, (y, z, x)))):
                    out[c] += diff(fn(*a))
    return out


_ODD = ((), (), (), (0, 1), (0, 2), (1, 2))


class _Demag:
    """h = -mu0 N * M on padded grids, leading dimensions being batches.  The
    transforms are products with the Fourier matrices, so that nothing rests
    on an FFT library."""

    def __init__(self, n, cell, box=(0, 0, 0), reps=(0, 0, 0)):
        self.n, self.pad = n, [2 * k if k > 1 else 1 for k in n]
        octant = _newell(n, cell, box, reps)
        full = torch.zeros((6, self.pad[2], self.pad[1], self.pad[0]), dtype=torch.float64, device=DEV)
        full[:, :n[2], :n[1], :n[0]] = octant
        for c in range(6):
            for a in range(3):
                if n[a] > 1:  # offsets -d at pad - d
                    d = 2 - a
                    neg = full[c].narrow(d, 1, n[a] - 1).flip(d) * (-1.0 if a in _ODD[c] else 1.0)
                    full[c].narrow(d, n[a] + 1, n[a] - 1).copy_(neg)

        def matrix(p, rows, cols, sign):
            jk = torch.outer(torch.arange(rows, device=DEV), torch.arange(cols, device=DEV)) % p
            w = 2 * math.pi / p * jk.double()
            return torch.complex(torch.cos(w), sign * torch.sin(w))

        px, py, pz = self.pad
        hx = px // 2 + 1
        self.fwd = [matrix(px, n[0], hx, -1), matrix(py, py, n[1], -1), matrix(pz, pz, n[2], -1)]
        weight = torch.full((hx, 1), 2.0, dtype=torch.float64, device=DEV)
        weight[0] = 1.0
        if px % 2 == 0:
            weight[-1] = 1.0
        self.inv = [weight * matrix(px, hx, n[0], 1) / px, matrix(py, n[1], py, 1) / py, matrix(pz, n[2], pz, 1) / pz]
        self.spec = torch.stack([self.transform(full[c], [matrix(px, px, hx, -1), matrix(py, py, py, -1),
                                                          matrix(pz, pz, pz, -1)], (0, 1, 2)) for c in range(6)])

    @staticmethod
    def transform(v, F, order):
        v = v.to(torch.complex128)
        for a in order:
            if a == 0:
                v = torch.matmul(v, F[0])
            elif a == 1:
                v = torch.matmul(F[1], v)
            else:
                flat = v.reshape(*v.shape[:-3], v.shape[-3], -1)
                v = torch.matmul(F[2], flat).reshape(*v.shape[:-3], F[2].shape[0], *v.shape[-2:])
        return v

    def __call__(self, M):
        v = self.transform(M, self.fwd, (0, 1, 2))
        xx, yy, zz, xy, xz, yz = self.spec
        a, b, c = v[..., 0, :, :, :], v[..., 1, :, :, :], v[..., 2, :, :, :]
        h = torch.stack((xx * a + xy * b + xz * c, xy * a + yy * b + yz * c, xz * a + yz * b + zz * c), dim=-4)
        return -MU0 * self.transform(h, self.inv, (2, 1, 0)).real


def _f32(v):
    return float(np.float32(v))


def _cross(a, b):
    return torch.cross(a, b, dim=-4)


def _dot(a, b):
    return (a * b).sum(-4, keepdim=True)


def _stack(x, y, z):
    return torch.stack((x, y, z), dim=-4)


def _comp(v):
    return v[..., 0, :, :, :], v[..., 1, :, :, :], v[..., 2, :, :, :]


class _Grid:
    """Neighbours of every cell along an axis, with the mask of those present."""

    def __init__(self, n, cell, periodic=(False, False, False), geom=None):
        self.n, self.cell, self.periodic = n, cell, periodic
        self.geom = torch.ones((n[2], n[1], n[0]), dtype=torch.bool, device=DEV) if geom is None else geom
        self.has = {(a, s): self.shift(self.geom, a, s) & self.inside(a, s) for a in range(3) for s in (-1, 1)}

    def shift(self, v, a, s):
        return torch.roll(v, -s, -1 - a)

    def inside(self, a, s):
        ok = torch.ones(self.n[a], dtype=torch.bool, device=DEV)
        if not self.periodic[a]:
            ok[-1 if s > 0 else 0] = False
        return ok.reshape([-1 if d == 2 - a else 1 for d in range(3)])


def _gamma(D, a, m):
    """The DMI boundary vector of axis a: D[a] = (xy, xz, yz)."""
    xy, xz, yz = D[a]
    x, y, z = _comp(m)
    return _stack(-xy * y - xz * z, xy * x - yz * z, xz * x + yz * y)


def _harm(a, b):
    return torch.where(a + b != 0, 2 * a * b / torch.where(a + b != 0, a + b, 1.0), 0.0) if torch.is_tensor(a) else a


def _interfacial(d):
    return ((0.0, d, 0.0), (0.0, 0.0, d), (0.0, 0.0, 0.0))


class _Ferro:
    """Fields of one or more (leading dimension) ferromagnets, 64 bits."""

    def __init__(self, grid, demag, msat, aex, alpha, D=None, ku=None, bias=0.0, jcur=0.0):
        self.g, self.demag, self.ms, self.a, self.alpha, self.D = grid, demag, msat, aex, alpha, D
        self.ku, self.bias, self.jcur = ku, bias, jcur

    def terms(self, m):
        g = self.g
        hex_, hdm = torch.zeros_like(m), torch.zeros_like(m)
        for (ax, s), has in g.has.items():
            if g.n[ax] == 1 and not g.periodic[ax] and (self.D is None or not any(self.D[ax])):
                continue
            mn = g.shift(m, ax, s)
            if self.D is not None:
                mn = torch.where(has, mn, m + s * g.cell[ax] / (2 * self.a) * _gamma(self.D, ax, m))
                hdm = hdm - (s / g.cell[ax]) * _gamma(self.D, ax, mn)
            else:
                mn = torch.where(has, mn, m)
            hex_ = hex_ + 2 * self.a / g.cell[ax] ** 2 * (mn - m)
        out = {"ex": hex_ / self.ms, "dm": hdm / self.ms}
        if self.ku is not None:
            z = torch.zeros_like(m)
            z[..., 2, :, :, :] = (2 * self.ku / self.ms * m[..., 2:3, :, :, :])[..., 0, :, :, :]
            out["an"] = z
        if self.bias:
            b = torch.zeros_like(m)
            b[..., 0, :, :, :] = self.bias
            out["ext"] = b
        out["demag"] = self.demag(self.ms * m)
        return {k: torch.where(g.geom, v, 0.0) for k, v in out.items()}

    def rhs(self, m):
        h = sum(self.terms(m).values())
        mxh = _cross(m, h)
        t = -GAMMA / (1 + self.alpha ** 2) * (mxh + self.alpha * _cross(m, mxh))
        if self.jcur:
            g, xi, pol, al = self.g, 0.2, 0.6, self.alpha
            u = MUB * pol / (QE * self.ms * (1 + xi * xi)) * self.jcur
            hs = torch.zeros_like(m)
            for s in (-1, 1):
                hs = hs + torch.where(g.inside(0, s), s * u / (2 * g.cell[0]) * g.shift(m, 0, s), 0.0)
            mxs = _cross(m, hs)
            t = t - ((1 + xi * al) * _cross(m, mxs) + (xi - al) * mxs) / (1 + al * al)
        return torch.where(self.g.geom, t, 0.0)

    def energy(self, m):
        e, t = 0.0, self.terms(m)
        for k, f in (("ex", 0.5), ("dm", 0.5), ("demag", 0.5), ("ext", 1.0)):
            if k in t:
                e = e - f * (self.ms * _dot(m, t[k])).sum()
        if self.ku is not None:
            e = e - (self.ku * m[..., 2:3, :, :, :] ** 2).sum()
        return e * self.g.cell[0] * self.g.cell[1] * self.g.cell[2]


_TABLEAU = {
    "Heun": ([[], [1]], [1 / 2, 1 / 2]),
    "BogackiShampine": ([[], [1 / 2], [0, 3 / 4]], [2 / 9, 1 / 3, 4 / 9]),
    "Fehlberg": ([[], [1 / 4], [3 / 32, 9 / 32], [1932 / 2197, -7200 / 2197, 7296 / 2197],
                  [439 / 216, -8, 3680 / 513, -845 / 4104], [-8 / 27, 2, -3544 / 2565, 1859 / 4104, -11 / 40]],
                 [16 / 135, 0, 6656 / 12825, 28561 / 56430, -9 / 50, 2 / 55]),
    "DormandPrince": ([[], [1 / 5], [3 / 40, 9 / 40], [44 / 45, -56 / 15, 32 / 9],
                       [19372 / 6561, -25360 / 2187, 64448 / 6561, -212 / 729],
                       [9017 / 3168, -355 / 33, 46732 / 5247, 49 / 176, -5103 / 18656]],
                      [35 / 384, 0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84]),
}
# Dormand and Prince's error weights: fifth order minus the embedded fourth
_DP_ERR = [35 / 384 - 5179 / 57600, 0, 500 / 1113 - 7571 / 16695, 125 / 192 - 393 / 640,
           -2187 / 6784 + 92097 / 339200, 11 / 84 - 187 / 2100, -1 / 40]


def _unit(m):
    n = torch.sqrt(_dot(m, m))
    return torch.where(n > 0, m / torch.where(n > 0, n, 1.0), 0.0)


def _combine(x, k, c, h, unit):
    """x + h sum_j c_j k_j of every variable, the magnetisations normalised."""
    out = []
    for i, v in enumerate(x):
        for cj, kj in zip(c, k):
            if cj:
                v = v + h * cj * kj[i]
        out.append(_unit(v) if unit[i] else v)
    return out


def _step(rhs, x, h, method, unit, first=None):
    A, w = _TABLEAU[method]
    k = []
    for row in A:
        k.append(first if first is not None and not k else rhs(_combine(x, k, row, h, unit)))
    return _combine(x, k, w, h, unit), k


def _adaptive(rhs, x, duration):
    """The controller of the reference's time solver with Dormand-Prince."""
    unit, t = [True], 0.0
    first = rhs(x)
    norm = lambda v: float(torch.sqrt(_dot(v, v)).max())  # noqa: E731
    dt, last = 0.01 / norm(first[0]), False
    while not last:
        last = not t < duration - dt
        if last:
            dt = duration - t
        while True:
            y, k = _step(rhs, x, dt, "DormandPrince", unit, first)
            end = rhs(y)
            err = norm(sum(e * kk[0] for e, kk in zip(_DP_ERR, k + [end]))) * dt
            h, ok = dt, err < 1e-5
            dt *= min(2.0, max(0.5, 0.8 * (1e-5 / max(err, 1e-300)) ** (1 / 6 if ok else 1 / 5)))
            if ok:
                break
        x, first, t = y, end, t + h
    return x


def _tensor(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV).double()


def _state(m0, geom=None):
    """The magnetisation as an assignment stores it: normalised, in 32 bits."""
    m = _unit(_tensor(m0)).float().double()
    return m if geom is None else torch.where(geom, m, 0.0)


def _ferro_of(case, seed):
    m0, geom, msat, ku = _llg_inputs(case, seed)
    n = (case["nx"], case["ny"], case["nz"])
    cell = tuple(_f32(c) for c in (case["cell"], case["cell"], case["cz"]))
    per = (bool(case["pbc"]),) * 2 + (False,)
    g = None if geom is None else torch.from_numpy(geom).to(DEV)
    box, reps = ((n[0], n[1], 0), (case["pbc"],) * 2 + (0,)) if case["pbc"] else ((0, 0, 0), (0, 0, 0))
    val = lambda v: _tensor(v) if isinstance(v, np.ndarray) else _f32(v)  # noqa: E731
    fm = _Ferro(_Grid(n, cell, per, g), _Demag(n, cell, box, reps), val(msat), _f32(case["aex"]), _f32(case["alpha"]),
                _interfacial(_f32(case["dmi"])) if case["dmi"] else None, val(ku) if case["ku"] else None,
                _f32(case["bias"]), _f32(case["jcur"]))
    return fm, _state(m0, g)


def _exact_afm(case, seed):
    m1, m2, u0 = _afm_inputs(case, seed)
    nx, ny = case["nx"], case["ny"]
    p = {k: _f32(v) if k not in ("reps", "dt") else v for k, v in _AFM.items()}
    c = _f32(2e-9)
    n, cell = (nx, ny, 1), (c, c, c)
    g = _Grid(n, cell, (True, True, False))
    demag = _Demag(n, cell, (nx, ny, 0), (p["reps"], p["reps"], 0))
    d, A, ms, al = p["dmi"], p["aex"], p["msat"], p["alpha"]
    D = ((0.0, 0.0, d), (0.0, -d, 0.0), (d, 0.0, 0.0))  # bulk, rows (xy, xz, yz) per axis
    el = case["elastic"]

    def deriv(v, a):  # fourth-order central difference, periodic; nothing along a single layer
        s = lambda k: torch.roll(v, -k, -1 - a)  # noqa: E731
        return (2 / 3 * (s(1) - s(-1)) + 1 / 12 * (s(-2) - s(2))) / cell[a]

    def inter(a, v):
        xy, xz, yz = D[a]
        x, y, z = _comp(v)
        return _stack(xy * y - xz * z, -xy * x - yz * z, -xz * x + yz * y)

    def field(m, s):
        h = torch.zeros_like(m)
        for (a, sg), has in g.has.items():
            mn, sn = g.shift(m, a, sg), g.shift(s, a, sg)
            if a == 2:  # free surfaces
                mn = m + sg * cell[a] / (2 * A) * _gamma(D, a, m)
                sn = s + sg * cell[a] / (2 * A) * _gamma(D, a, s)
            h = h + 2 * A / cell[a] ** 2 * (mn - m)
            h = h - sg / cell[a] * (_gamma(D, a, mn) + inter(a, sn))
        return h / ms + 4 * p["afmex_cell"] / (p["latcon"] ** 2 * ms) * s

    def rhs(x):
        a, b = x[0], x[1]
        hd = demag(ms * a + ms * b)
        if el:
            ux, uy = deriv(x[2], 0), deriv(x[2], 1)
            exx, eyy, exy = ux[0], uy[1], 0.5 * (ux[1] + uy[0])
            exz, eyz, ezz = 0.5 * ux[2], 0.5 * uy[2], torch.zeros_like(ux[0])
        out = []
        for m, s in ((a, b), (b, a)):
            h = field(m, s) + hd
            if el:
                X, Y, Z = m
                h = h - 2 / ms * p["B"] * _stack(exx * X + exy * Y + exz * Z, eyy * Y + eyz * Z + exy * X,
                                                 ezz * Z + exz * X + eyz * Y)
            mxh = _cross(m, h)
            out.append(-GAMMA / (1 + al * al) * (mxh + al * _cross(m, mxh)))
        if el:
            c11, c12, c44 = p["C11"], p["C12"], p["C44"]
            sxx, syy = c11 * exx + c12 * (eyy + ezz), c11 * eyy + c12 * (exx + ezz)
            sxy, sxz, syz = 2 * c44 * exy, 2 * c44 * exz, 2 * c44 * eyz
            f = deriv(_stack(sxx, sxy, sxz), 0) + deriv(_stack(sxy, syy, syz), 1)
            for m in (a, b):
                dx, dy = deriv(m, 0), deriv(m, 1)
                X, Y, Z = m
                f = f + p["B"] * _stack(2 * X * dx[0] + X * dy[1] + Y * dy[0], 2 * Y * dy[1] + Y * dx[0] + X * dx[1],
                                        Z * (dx[0] + dy[1]) + X * dx[2] + Y * dy[2])
            out += [x[3], (f - p["eta"] * x[3]) / p["rho"]]
        return out

    x = [_state(m1), _state(m2)] + ([_tensor(u0), torch.zeros_like(_tensor(u0))] if el else [])
    unit = [True, True, False, False][:len(x)]
    for _ in range(case["steps"]):
        x, _ = _step(rhs, x, p["dt"], "DormandPrince", unit)
    return x


def _exact_batch(case, seed):
    specs = _batch_inputs(case, seed)
    out, groups = [None] * len(specs), {}
    for i, (size, _, _) in enumerate(specs):
        groups.setdefault(size, []).append(i)
    cell = (_f32(2e-9),) * 3
    for size, ids in groups.items():
        col = lambda k: torch.tensor([specs[i][1][k] for i in ids], dtype=torch.float64,  # noqa: E731
                                     device=DEV).reshape(-1, 1, 1, 1, 1)
        fm = _Ferro(_Grid(size, cell), _Demag(size, cell), col("msat"), col("aex"), col("alpha"), ku=col("ku1"))
        x = [torch.stack([_state(specs[i][2]) for i in ids])]
        for _ in range(case["steps"]):
            x, _ = _step(lambda v: [fm.rhs(v[0])], x, _BATCH_DT, "DormandPrince", [True])
        for j, i in enumerate(ids):
            out[i] = x[0][j].reshape(-1)
    per = -(-len(out) // 32)
    return [torch.cat(out[i:i + per]) for i in range(0, len(out), per)]


def exact(case, seed):
    kind = case["kind"]
    if kind == "afm":
        return _exact_afm(case, seed)
    if kind == "batch":
        return _exact_batch(case, seed)
    if kind == "demag":
        g = torch.Generator(device=DEV).manual_seed(seed)
        shape = (case["nz"], case["ny"], case["nx"])
        m = torch.randn((3,) + shape, generator=g, device=DEV)
        m /= m.norm(dim=0)
        n, c = (case["nx"], case["ny"], case["nz"]), 4e-9
        box, reps = ((n[0], n[1], 0), (case["pbc"],) * 2 + (0,)) if case["pbc"] else ((0, 0, 0), (0, 0, 0))
        mask = torch.from_numpy(_disk(shape)).to(DEV) if case["geom"] else torch.ones(shape, dtype=torch.bool, device=DEV)
        h = _Demag(n, (c, c, c), box, reps)(torch.where(mask, 8e5 * m.double(), 0.0))
        return torch.where(mask, h, 0.0)
    if kind == "table":
        case = _llg(nx=case["nx"], ny=case["ny"], nz=case["nz"], steps=2, dt=1e-13, alpha=0.1, bias=0.02, ku=1e5)
    fm, m = _ferro_of(case, seed)
    x = [m]
    rhs = lambda v: [fm.rhs(v[0])]  # noqa: E731
    if case["duration"]:
        x = _adaptive(rhs, x, case["duration"])
    else:
        for _ in range(case["steps"]):
            x, _ = _step(rhs, x, case["dt"], case["method"], [True])
    m = x[0]
    if kind == "llg":
        return m
    t = fm.terms(m)
    h = sum(t.values())
    return {"average": m.reshape(3, -1).mean(1), "energy": float(fm.energy(m)), "torque":
            float(torch.sqrt(_dot(fm.rhs(m), fm.rhs(m))).max()), "demag": t["demag"], "field": h, "m": m}
