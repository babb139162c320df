"""The direct demag sum of small grids, and the one-launch evaluation on it.

Grids at the edges of the strips (four x cells), of the wavefronts per strip
and of the rule that chooses the sum, against the FP64 oracle: field error at
most 4e-7 of the largest field (FP32 kernel and products, short chains).  The
same magnets' torque, which one launch forms with the field, against the
torque formed from the demag field in memory by the per-cell kernel.
"""

import numpy as np
import pytest

from helpers import make_pair, random_unit
from oracle import demag as odemag

import mumaxplus as mp

pytestmark = pytest.mark.gpu

# 641 cells and more are summed, as far as the rule goes (test_rule): the last
# three and 2 x 350 x 3 lie on its other side.  No axis is longer than 350 cells: the FP64 tensor's own cancellation
# (27 terms of r^3 2^-53 / (4 pi) at r cells) is 1e-8 there, but 8e-8 an entry
# at 700, which the oracle and the device round differently.
SIZES = [(214, 3, 1), (3, 214, 1), (2, 2, 161), (64, 64, 1), (257, 3, 1), (128, 32, 1), (43, 15, 1), (2, 350, 3),
         (33, 9, 4), (16, 16, 14), (64, 65, 1), (32, 16, 8), (32, 20, 1)]


def _grid(size):
    nx, ny, nz = size
    rng = np.random.default_rng(nx + 7 * ny + 31 * nz)
    m = random_unit(rng, (nz, ny, nx)).astype(np.float32)
    return rng, m


@pytest.mark.parametrize("size", SIZES)
def test_field(size):
    rng, m = _grid(size)
    nx, ny, nz = size
    cs = (3e-9, 2e-9, 4e-9)
    world = mp.World(cs)
    geom = rng.random((nz, ny, nx)) > 0.2 if nx * ny * nz > 20 else None
    mag = mp.Ferromagnet(world, mp.Grid(size), geometry=geom)
    ms = (8e5 * rng.uniform(0.5, 1.5, (nz, ny, nx))).astype(np.float32)
    mag.msat = ms
    mag.magnetization = m
    want = odemag.demag_fft(mag.magnetization.get().astype(float), ms.astype(float), world.cellsize, geom)
    got = mag.demag_field()
    assert np.abs(got - want).max() <= 4e-7 * np.abs(want).max()


@pytest.mark.parametrize("pbc", [(1, 0, 0), (2, 1, 0)])
def test_periodic(pbc):
    size = (38, 11, 2)
    _, m = _grid(size)
    cs = (3e-9, 2e-9, 4e-9)
    box = tuple(n if p else 0 for n, p in zip(size, pbc))
    world = mp.World(cs, mastergrid=mp.Grid(box), pbc_repetitions=pbc)
    mag = mp.Ferromagnet(world, mp.Grid(size))
    mag.msat = 8e5
    mag.magnetization = m
    want = odemag.demag_fft(mag.magnetization.get().astype(float), 8e5, world.cellsize, None, box, pbc)
    assert np.abs(mag.demag_field() - want).max() <= 4e-7 * np.abs(want).max()


@pytest.mark.parametrize("size", [(51, 13, 1), (64, 64, 1), (33, 9, 4), (16, 16, 14)])
@pytest.mark.parametrize("kind", ["uniform", "uniform parameters", "per cell"])
def test_stepped_torque(size, kind):
    """One fixed Heun step takes two one-launch evaluations; the oracle's step is the reference."""
    rng, m = _grid(size)
    nx, ny, nz = size
    p = {"msat": 8e5, "aex": 1.3e-11, "alpha": 0.05, "ku1": 3e5, "anisU": (0, 0.6, 0.8)}
    if kind == "uniform parameters":
        p.update(jcur=(1e12, 0, 0), xi=0.1, pol=0.5)
    if kind == "per cell":
        p["ku1"] = (3e5 * rng.uniform(0.5, 1.5, (nz, ny, nx))).astype(np.float32)
    world, mag, ow, om = make_pair(size, (3e-9, 2e-9, 4e-9), p, m, geometry=rng.random((nz, ny, nx)) > 0.2)
    for ts in (world.timesolver, ow.solver):
        ts.set_method("Heun")
    world.timesolver.adaptive_timestep, world.timesolver.timestep = False, 2e-14
    ow.solver.adaptive, ow.solver.dt = False, 2e-14
    m0 = mag.magnetization.get().astype(float)
    world.timesolver.steps(1)
    ow.solver.steps(1)
    dm, want = mag.magnetization.get() - m0, om.m - m0
    # the step moves m by up to a few percent: its error is that of m (2^-24) over the move
    assert np.abs(dm - want).max() <= 1e-5 * np.abs(want).max() + 1.5e-7


def test_two_sublattices():
    """Ms1 m1 + Ms2 m2 as the source."""
    size = (33, 25, 1)
    rng, m = _grid(size)
    world = mp.World((3e-9, 2e-9, 4e-9))
    afm = mp.Antiferromagnet(world, mp.Grid(size))
    afm.sub1.msat, afm.sub2.msat = 6e5, 3e5
    afm.sub1.magnetization = m
    afm.sub2.magnetization = random_unit(rng, size[::-1]).astype(np.float32)
    M = 6e5 * afm.sub1.magnetization.get().astype(float) + 3e5 * afm.sub2.magnetization.get().astype(float)
    want = odemag.demag_fft(M, 1.0, world.cellsize)
    assert np.abs(afm.sub1.demag_field() - want).max() <= 4e-7 * np.abs(want).max()


# Grids at the edges of the rule (strips of four x cells: 1024, rows of two to
# four cells 768, rows of one cell none), and whether they are summed.
RULE = [((64, 64, 1), True), ((13, 256, 1), True), ((5, 256, 4), False), ((5, 16, 32), True), ((5, 171, 3), False),
        ((4, 256, 3), True), ((4, 193, 4), False), ((2, 32, 24), True), ((2, 350, 3), False), ((1, 30, 100), False),
        ((1, 55, 55), False), ((1, 350, 2), False), ((641, 1, 1), True), ((32, 20, 1), False), ((65, 64, 1), False)]


@pytest.mark.parametrize("size,direct", RULE)
def test_rule(size, direct):
    nx, ny, nz = size
    _, m = _grid(size)
    world = mp.World((3e-9, 2e-9, 4e-9))
    mag = mp.Ferromagnet(world, mp.Grid(size))
    mag.msat, mag.aex, mag.alpha = 8e5, 1.3e-11, 0.1
    mag.magnetization = m
    want = odemag.demag_fft(mag.magnetization.get().astype(float), 8e5, world.cellsize)
    tol = 6e-7 + 3e-15 * max(size) ** 3  # the passes' rounding and the FP64 tensor's own, as for few layers
    assert np.abs(mag.demag_field() - want).max() <= tol * np.abs(want).max()
    world.timesolver.adaptive_timestep, world.timesolver.timestep = False, 1e-15
    world.timesolver.steps(1)
    impl = world._impl
    impl.set_profiling(True)
    impl.profile_reset()
    world.timesolver.steps(1)
    names = set(impl.profile_report())
    impl.set_profiling(False)
    assert ("k_xfwd" in names) == (not direct), names


@pytest.mark.parametrize("size", [(1, 1024, 3), (3, 1024, 1), (1, 30, 100), (13, 256, 1), (1000, 4, 1), (6, 256, 2)])
def test_most_strips(size):
    """Long and narrow grids, on both sides of the rule: a field that is not zero and equals its mirror image."""
    rng, m = _grid(size)
    world = mp.World((3e-9, 2e-9, 4e-9))
    mag = mp.Ferromagnet(world, mp.Grid(size))
    mag.msat = 8e5
    mag.magnetization = m
    h = mag.demag_field()
    flip = mag.magnetization.get()[:, ::-1, ::-1, ::-1].copy()
    mag.magnetization = flip
    assert np.abs(h).max() > 0.01
    # a point reflection of the source reflects the field; the sums run in another order
    assert np.abs(mag.demag_field()[:, ::-1, ::-1, ::-1] - h).max() <= 1e-6 * np.abs(h).max()
