"""The uniform field kernel's extended instances against the FP64 oracle: per-cell
Ms (cells without moment among them) and Ku1, and the Zhang-Li torque, with and
without a mask, periodic axes and DMI, on rows that are no multiple of a block
and on the grids that are summed directly; and the neighbouring parameter sets
that stay on the per-cell kernel (per-cell A, both together, A = 0)."""

import numpy as np
import pytest

from helpers import make_pair, random_unit

pytestmark = pytest.mark.gpu

SIZES = [(70, 61, 1), (33, 9, 3), (9, 5, 1), (1, 7, 2)]


def _step(size, params, dmi=None, **kw):
    rng = np.random.default_rng(sum(size))
    nx, ny, nz = size
    m = random_unit(rng, (nz, ny, nx)).astype(np.float32)
    p = {"msat": 8e5, "aex": 1.3e-11, "alpha": 0.05, "ku1": 3e5, "anisU": (0, 0.6, 0.8)}
    p.update(params(rng, (nz, ny, nx)))
    world, mag, ow, om = make_pair(size, (3e-9, 2e-9, 4e-9), p, m, dmi=dmi, world_bias=(0.01, 0.0, -0.02), **kw)
    world.timesolver.set_method("Heun")
    ow.solver.set_method("Heun", defer_timestep=True)
    world.timesolver.adaptive_timestep, world.timesolver.timestep = False, 1e-14
    ow.solver.adaptive, ow.solver.dt = False, 1e-14
    m0 = mag.magnetization.get().astype(float)
    world.timesolver.steps(1)
    ow.solver.steps(1)
    dm, want = mag.magnetization.get() - m0, om.m - m0
    # FP32 fields of 1e-5 over the move, and m's own last bit
    assert np.abs(dm - want).max() <= 1e-5 * np.abs(want).max() + 1.5e-7


def _cells(rng, shape):
    ms = 8e5 * rng.uniform(0.7, 1.3, shape)
    ms[rng.random(shape) < 0.1] = 0.0
    return {"msat": ms, "ku1": 3e5 * rng.uniform(0.5, 1.5, shape)}


VARIANTS = {
    "Ms and Ku1": _cells,
    "Ku1": lambda rng, shape: {"ku1": 3e5 * rng.uniform(0.5, 1.5, shape), "ku2": 1e5},
    "Zhang-Li": lambda rng, shape: {"jcur": (2e13, -1e13, 5e12), "xi": 0.1, "pol": 0.5},
    "per-cell A": lambda rng, shape: {"aex": 1.3e-11 * rng.uniform(0.7, 1.3, shape), **_cells(rng, shape)},
    "Ms and Zhang-Li": lambda rng, shape: {"jcur": (2e13, 0, 0), "xi": 0.1, "pol": 0.5, **_cells(rng, shape)},
    "no A": lambda rng, shape: {"aex": 0.0, **_cells(rng, shape)},
}


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("variant", VARIANTS)
def test_open(variant, size):
    _step(size, VARIANTS[variant])


@pytest.mark.parametrize("variant", ["Ms and Ku1", "Zhang-Li"])
def test_masked_periodic_dmi(variant):
    size = (70, 11, 2)
    geom = np.random.default_rng(3).random(size[::-1]) > 0.2
    dmi = {"xxz": 2e-3, "yyz": 2e-3}
    _step(size, VARIANTS[variant], dmi=dmi, geometry=geom)
    _step(size, VARIANTS[variant], dmi=dmi, mastergrid=(70, 0, 2), pbc=(1, 0, 1))
