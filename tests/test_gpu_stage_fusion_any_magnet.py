"""Stage combinations fused into the field launch for every magnet and tableau.

The field launch of a lone ferromagnet also forms the next stage state, and
with a tableau whose last stage is not the new state (Heun, Fehlberg,
CashKarp) the step's last field launch forms the final state.  The arithmetic
is that of the separate combination, so a fused run equals the unfused one
("fuse_stages" off) bit for bit: uniform magnets with and without a mask, and
magnets on the per-cell kernel (per-cell parameters, a spin-transfer torque,
regions), fixed and adaptive with rejected steps.
"""

import numpy as np
import pytest

from helpers import random_unit

import mumaxplus as mp

pytestmark = pytest.mark.gpu

KINDS = ("uniform", "masked", "grains", "stt", "regions")


def _world(kind, size, fuse, method):
    nx, ny, nz = size
    rng = np.random.default_rng(11)
    world = mp.World((2e-9, 2.5e-9, 3e-9))
    kw = {}
    if kind in ("masked", "grains"):
        kw["geometry"] = rng.random((nz, ny, nx)) > 0.15
    if kind == "regions":
        kw["regions"] = rng.integers(0, 2, (nz, ny, nx))
    mag = mp.Ferromagnet(world, mp.Grid(size), **kw)
    mag.msat, mag.aex, mag.alpha, mag.ku1, mag.anisU = 8e5, 1.3e-11, 0.05, 3e5, (0.1, 0.2, 1.0)
    mag.dmi_tensor.set_interfacial_dmi(2e-3)
    if kind == "grains":
        mag.msat = (8e5 * rng.uniform(0.8, 1.2, (1, nz, ny, nx))).astype(np.float32)
    if kind == "stt":
        mag.jcur, mag.xi, mag.pol = (1e12, 2e11, 0), 0.1, 0.5
    if kind == "regions":
        mag.inter_exchange = 4e-12
    mag.magnetization = random_unit(rng, (nz, ny, nx)).astype(np.float32)
    world._impl.set_option("fuse_stages", int(fuse))
    world.timesolver.set_method(method)
    return world, mag


@pytest.mark.parametrize("method", ["Heun", "BogackiShampine", "Fehlberg", "CashKarp", "DormandPrince"])
@pytest.mark.parametrize("kind", KINDS)
def test_fixed_steps(kind, method):
    out = []
    for fuse in (True, False):
        world, mag = _world(kind, (33, 14, 2), fuse, method)
        ts = world.timesolver
        ts.adaptive_timestep, ts.timestep = False, 4e-14
        ts.steps(6)
        ts.timestep = 3e-14
        ts.steps(2)
        mag.magnetization = random_unit(np.random.default_rng(2), (2, 14, 33)).astype(np.float32)
        ts.run(1.3e-13)
        out.append((mag.magnetization.get(), ts.time))
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]


@pytest.mark.parametrize("method", ["Heun", "Fehlberg", "CashKarp"])
@pytest.mark.parametrize("kind", ["uniform", "grains"])
def test_adaptive_with_rejections(kind, method):
    out = []
    for fuse in (True, False):
        world, mag = _world(kind, (20, 9, 1), fuse, method)
        ts = world.timesolver
        ts.max_error = 1e-6
        ts.timestep = 2e-12  # far too large: the first attempts are rejected
        ts._impl.run(2e-12)
        out.append((mag.magnetization.get(), ts.time, ts._impl.nsteps, ts._impl.nrejected))
    assert out[0][3] > 0
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1:] == out[1][1:]
