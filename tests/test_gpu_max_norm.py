"""The step controller's error norm and the largest torque, which one launch
reduces and hands over through host memory: grids of one block, of exactly as
many cells as a block, and of more blocks than the launch holds; masked cells
left out; many calls in a row and two worlds in turn."""

import numpy as np
import pytest

import mumaxplus as mp

pytestmark = pytest.mark.gpu


def _magnet(size, seed, mask=False):
    nx, ny, nz = size
    rng = np.random.default_rng(seed)
    world = mp.World((2e-9, 2e-9, 2e-9))
    geom = rng.random((nz, ny, nx)) > 0.3 if mask else None
    mag = mp.Ferromagnet(world, mp.Grid(size), geometry=geom)
    mag.enable_demag = False
    mag.msat, mag.aex, mag.alpha = 8e5, 1.3e-11, 0.1
    mag.magnetization = rng.normal(size=(3, nz, ny, nx)).astype(np.float32)
    return world, mag


def _want(mag):
    t = mag.torque().astype(np.float64)
    return np.sqrt((t * t).sum(axis=0)).max()


@pytest.mark.parametrize("mask", [False, True])
@pytest.mark.parametrize("size", [(1, 2, 1), (16, 16, 1), (257, 1, 1), (700, 500, 1)])
def test_largest_torque(size, mask):
    world, mag = _magnet(size, sum(size), mask)
    for _ in range(3):
        assert mag.max_torque() == pytest.approx(_want(mag), rel=1e-6)


def test_two_worlds_in_turn():
    made = [_magnet((40 + 8 * i, 20, 1), i) for i in range(2)]
    for _, mag in made:
        assert mag.max_torque() == pytest.approx(_want(mag), rel=1e-6)
    for k in range(50):
        world, mag = made[k % 2]
        world.timesolver.adaptive_timestep = True
        world.timesolver.run(2e-14)
        assert mag.max_torque() == pytest.approx(_want(mag), rel=1e-6)
