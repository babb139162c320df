"""Batches of few-layer, thick and single-layer members on the GPU.

Two to eight layers take the y and z transforms in one pass, more layers take
them in three, and a batch may hold both beside single layers.  Every member
ends bit for bit where the same magnet ends alone (with the batch's kernels:
world options fuse_stages, field_zchunk and direct_demag 0), and the persistent
kernel, whose phases depend on which kinds are present, ends there too.
"""

import numpy as np
import pytest

from helpers import random_unit

import mumaxplus as mp

pytestmark = pytest.mark.gpu

THICK, THICK_SMALL = (12, 8, 9), (8, 8, 10)
SEVEN, EIGHT, TWO, FOUR = (20, 10, 7), (9, 12, 8), (20, 12, 2), (31, 17, 4)
LONG_Y, LONGER_Y, LONG_THICK = (16, 130, 2), (6, 300, 5), (5, 140, 11)
FLAT = (32, 16, 1)

SHORT = {"thick": [THICK], "640 cells": [THICK_SMALL], "seven and eight layers": [SEVEN, EIGHT],
         "lean": [TWO, FOUR], "few and flat": [TWO, FLAT, SEVEN], "few and thick": [FOUR, THICK, EIGHT],
         "all": [FLAT, THICK, TWO, SEVEN, THICK_SMALL, FOUR, EIGHT]}
LONG = {"long y": [LONG_Y], "longer y": [LONGER_Y], "long all": [FLAT, LONG_Y, LONG_THICK, TWO, LONGER_Y]}


def _magnet(size, seed):
    nx, ny, nz = size
    rng = np.random.default_rng(seed)
    world = mp.World((2e-9, 2e-9, 2e-9))
    geom = rng.random((nz, ny, nx)) > 0.1 if seed % 2 else None
    mag = mp.Ferromagnet(world, mp.Grid(size), geometry=geom)
    mag.msat, mag.aex, mag.alpha, mag.ku1, mag.anisU = 8e5, 1.3e-11, 0.05, 2e5, (0.3, 0, 1)
    mag.magnetization = random_unit(rng, (nz, ny, nx)).astype(np.float32)
    ts = world.timesolver
    ts.set_method("DormandPrince")
    ts.adaptive_timestep, ts.timestep = False, 1e-13
    return world, mag


def _batch(sizes, mode):
    batch = mp.Batch(sum(int(np.prod(s)) + 256 for s in sizes))
    batch.step_mode = mode
    made = [_magnet(s, i) for i, s in enumerate(sizes)]
    ids = [batch.add(mag, steps=12) for _, mag in made]
    while len(batch.finished()) < len(ids):
        batch.advance(4)
    path = batch.step_path()["last_path"]
    for i in ids:
        batch.remove(i)
    return [mag.magnetization.get() for _, mag in made], path


@pytest.mark.parametrize("name", [*SHORT, *LONG])
def test_members_end_where_they_end_alone(name):
    sizes = {**SHORT, **LONG}[name]
    got, path = _batch(sizes, "passes")
    assert path == "passes"
    for i, (size, m) in enumerate(zip(sizes, got)):
        world, mag = _magnet(size, i)
        for key in ("fuse_stages", "field_zchunk", "direct_demag"):
            world._impl.set_option(key, 0)
        world.timesolver.steps(12)
        assert np.array_equal(m, mag.magnetization.get()), size


@pytest.mark.parametrize("name", SHORT)
def test_persistent_equals_per_pass(name):
    want, _ = _batch(SHORT[name], "passes")
    got, path = _batch(SHORT[name], "persistent")
    assert path == "persistent"
    for size, a, b in zip(SHORT[name], got, want):
        assert np.array_equal(a, b), size


@pytest.mark.parametrize("mode", ["passes", "persistent"])
def test_reports_between_admission_and_steps(mode):
    """Reading the batch's reports after an admission leaves the new member's steps as they are."""
    sizes = [FLAT, TWO, SEVEN]
    out = []
    for ask in (False, True):
        batch = mp.Batch(8192)
        batch.step_mode = mode
        made = [_magnet(s, i) for i, s in enumerate(sizes)]
        ids = []
        for _, mag in made:
            ids.append(batch.add(mag, steps=6))
            if ask:
                assert batch.info()["step_bytes"] > 0 and batch.step_path()["persist_grid"] > 0
            batch.advance(2)
        while len(batch.finished()) < len(ids):
            batch.advance(2)
        for i in ids:
            batch.remove(i)
        out.append([mag.magnetization.get() for _, mag in made])
    for a, b in zip(*out):
        assert np.array_equal(a, b)
