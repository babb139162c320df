"""The demag pass of two to eight layers (y transforms and direct z sums in one
launch) against the FP64 oracle: every layer count, line lengths of 8 to 2048
points (lines of part of a wavefront to four of them), more lines than a block
transforms at a time, a mask, periodic images, and the layer counts and line
lengths just outside its rule."""

import numpy as np
import pytest

from helpers import DeviceBuffer, random_unit
from oracle import demag as odemag

import mumaxplus as mp

pytestmark = pytest.mark.gpu


# grids of more than 4096 cells, or of up to 640: others are summed directly
SIZES = [(150, 30, 2), (90, 20, 3), (70, 20, 4), (60, 15, 5), (50, 15, 6), (40, 17, 7), (40, 17, 8), (40, 15, 9),
         (700, 4, 2), (500, 3, 3), (3, 300, 5), (20, 129, 3), (17, 65, 6), (30, 257, 2), (9, 512, 4), (5, 513, 2),
         (5, 513, 3), (6, 5, 8), (1, 40, 3), (40, 1, 3)]
# long y lines, which take more than one round, on either side of the width
# from which they are one pass
SIZES += [(17, 300, 4), (16, 300, 4), (33, 270, 5), (17, 520, 2), (16, 520, 2), (9, 300, 2), (16, 140, 8)]


@pytest.mark.parametrize("size", SIZES)
def test_field(size):
    nx, ny, nz = size
    rng = np.random.default_rng(nx + 7 * ny + 31 * nz)
    world = mp.World((3e-9, 2e-9, 4e-9))
    geom = rng.random((nz, ny, nx)) > 0.2
    mag = mp.Ferromagnet(world, mp.Grid(size), geometry=geom)
    ms = (8e5 * rng.uniform(0.5, 1.5, (nz, ny, nx))).astype(np.float32)
    mag.msat = ms
    mag.magnetization = random_unit(rng, (nz, ny, nx)).astype(np.float32)
    want = odemag.demag_fft(mag.magnetization.get().astype(float), ms.astype(float), world.cellsize, geom)
    # FP32 transforms (a few 2^-24 of the largest field per pass), and the FP64
    # tensor's own cancellation at the far end of a long axis (r^3 2^-53, as
    # the oracle and the device round it differently)
    tol = 6e-7 + 3e-15 * max(size) ** 3
    assert np.abs(mag.demag_field() - want).max() <= tol * np.abs(want).max()


@pytest.mark.parametrize("pbc", [(1, 0, 0), (0, 2, 0), (2, 1, 0)])
def test_periodic(pbc):
    size = (80, 24, 3)
    box = tuple(n if p else 0 for n, p in zip(size, pbc))
    rng = np.random.default_rng(5)
    world = mp.World((3e-9, 2e-9, 4e-9), mastergrid=mp.Grid(box), pbc_repetitions=pbc)
    mag = mp.Ferromagnet(world, mp.Grid(size))
    mag.msat = 8e5
    mag.magnetization = random_unit(rng, size[::-1]).astype(np.float32)
    want = odemag.demag_fft(mag.magnetization.get().astype(float), 8e5, world.cellsize, None, box, pbc)
    assert np.abs(mag.demag_field() - want).max() <= 6e-7 * np.abs(want).max()


# line pairs on either side of the block size rule of the long x lines
# (1024 points: 384 pairs, 2048 points: 128 pairs)
@pytest.mark.parametrize("size", [(300, 256, 1), (300, 257, 1), (260, 128, 2), (520, 85, 1), (520, 86, 1)])
def test_long_x_lines(size):
    test_field(size)


def _length(n):
    k = 8
    while k < 2 * n - 1:
        k *= 2
    return 1 if n == 1 else k


@pytest.mark.parametrize("size", [(70, 33, 4), (300, 20, 1), (64, 64, 1), (33, 9, 4), (20, 30, 9), (17, 300, 4),
                                  (16, 300, 4), (17, 520, 2), (16, 520, 2), (9, 300, 2), (16, 140, 8)])
def test_plan_memory(size):
    """A plan holds the tables that its field needs, and reports them with its intermediates."""
    nx, ny, nz = size
    kx, ky, kz = (_length(n) for n in size)
    hx, hy, hz = kx // 2 + 1, ky // 2 + 1, kz // 2 + 1
    few = 2 <= nz <= 8 and size not in ((16, 300, 4), (16, 520, 2))
    # (x, y) spectra of every layer distance, or the whole spectrum: 6 floats an entry
    tables = 24 * hx * hy * (nz if few else hz)
    if size in ((64, 64, 1), (33, 9, 4)):  # summed directly: 4 (or 6) floats for dx from -4 nb to 4 nb
        tables += (16 if nz == 1 else 24) * ny * nz * 8 * ((nx + 3) // 4)
    plan = mp._cpp.DemagPlan(size, (3e-9, 2e-9, 4e-9))
    assert plan.info()[2] == tables
    m, h = DeviceBuffer(12 * nx * ny * nz), DeviceBuffer(12 * nx * ny * nz)
    plan.exec(m.ptr, h.ptr)
    a, b = 24 * nz * hx * ny, 0 if nz == 1 or few else 24 * hx * ky * nz
    assert plan.info()[2] == tables + a + b
