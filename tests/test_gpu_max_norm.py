"""The step controller's error norm and the largest torque, which one launch
reduces and hands over through host memory: grids of one block, of exactly as
many cells as a block, and of more blocks than the launch holds; masked cells
left out; many calls in a row and two worlds in turn; more worlds than one page
of host words serves, and again after they have gone."""

import gc

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


def test_more_worlds_than_a_page_of_words():
    for total in (1100, 3, 520):
        made = []
        for i in range(total):
            world = mp.World((2e-9, 2e-9, 2e-9))
            mag = mp.Ferromagnet(world, mp.Grid((2, 1, 1)))
            mag.enable_demag = False
            # two cells tilted by an angle of their own: the field along z turns each
            mag.msat, mag.alpha = 8e5, 0.1
            world.bias_magnetic_field = (0.0, 0.0, 1e-3 * (i + 1))
            mag.magnetization = (1.0, 0.0, 0.0)
            made.append((world, mag))
            assert mag.max_torque() > 0
        # m along x, B along z: |torque| = gamma B / sqrt(1 + alpha^2)
        want = 1.7595e11 / np.sqrt(1.01) * 1e-3 * np.arange(1, total + 1)
        got = np.array([mag.max_torque() for _, mag in made])
        assert np.abs(got / want - 1).max() < 1e-6
        for _, mag in made[::2]:
            assert mag.max_torque() > 0
        del world, mag, made
        gc.collect()
