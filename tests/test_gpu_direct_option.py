"""The world option "direct_demag": off, a small magnet's demag field comes from
the FFT passes again, in its quantities, its steps and those of an
antiferromagnet, and (with fuse_stages and field_zchunk 0) its steps equal its
steps in a batch bit for bit."""

import numpy as np
import pytest

from helpers import random_unit

import mumaxplus as mp

pytestmark = pytest.mark.gpu

CS = (2e-9, 2e-9, 2e-9)


def _magnet(size, seed=1):
    nx, ny, nz = size
    world = mp.World(CS)
    mag = mp.Ferromagnet(world, mp.Grid(size))
    mag.msat, mag.aex, mag.alpha, mag.ku1, mag.anisU = 8e5, 1.3e-11, 0.05, 2e5, (0, 0, 1)
    mag.magnetization = random_unit(np.random.default_rng(seed), (nz, ny, nx)).astype(np.float32)
    ts = world.timesolver
    ts.set_method("DormandPrince")
    ts.adaptive_timestep, ts.timestep = False, 1e-13
    return world, mag


# on both sides of the direct sum's range
@pytest.mark.parametrize("size", [(33, 17, 1), (40, 24, 1), (64, 64, 1), (30, 15, 3), (16, 16, 14), (70, 64, 1)])
def test_steps_equal_the_batch_bit_for_bit(size):
    bw, bm = _magnet(size)
    batch = mp.Batch(8192)
    batch.add(bm, steps=30)
    batch.run_until_done()
    world, mag = _magnet(size)
    for key in ("fuse_stages", "field_zchunk", "direct_demag"):
        world._impl.set_option(key, 0)
        assert world._impl.get_option(key) == 0
    world.timesolver.steps(30)
    assert np.array_equal(mag.magnetization.get(), bm.magnetization.get())


def _kernels(world, work):
    impl = world._impl
    impl.set_profiling(True)
    impl.profile_reset()
    work()
    rep = impl.profile_report()
    impl.set_profiling(False)
    return set(rep)


def test_launches_and_fields():
    world, mag = _magnet((40, 24, 1))
    assert world._impl.get_option("direct_demag") == 1
    want = mag.demag_field()
    world._impl.set_option("direct_demag", 0)
    # 4e-7 of the largest field each against 64 bits
    assert np.abs(mag.demag_field() - want).max() <= 8e-7 * np.abs(want).max() and np.abs(want).max() > 0
    for direct in (0, 1):
        world._impl.set_option("direct_demag", direct)
        assert ("k_xfwd" in _kernels(world, lambda: world.timesolver.steps(2))) == (not direct)


def test_antiferromagnet():
    world = mp.World(CS)
    afm = mp.Antiferromagnet(world, mp.Grid((40, 24, 1)))
    afm.msat, afm.aex, afm.alpha = 6e5, 5e-12, 0.1
    for s, seed in ((afm.sub1, 1), (afm.sub2, 2)):
        s.enable_demag = True
        s.magnetization = random_unit(np.random.default_rng(seed), (1, 24, 40)).astype(np.float32)
    world.timesolver.adaptive_timestep, world.timesolver.timestep = False, 1e-15
    want = afm.sub1.demag_field()
    world._impl.set_option("direct_demag", 0)
    assert np.abs(afm.sub1.demag_field() - want).max() <= 8e-7 * np.abs(want).max() and np.abs(want).max() > 0
    for direct in (0, 1):
        world._impl.set_option("direct_demag", direct)
        k = _kernels(world, lambda: world.timesolver.steps(1))
        assert ("k_direct" in k) == bool(direct) and ("k_xfwd" in k) == (not direct)
