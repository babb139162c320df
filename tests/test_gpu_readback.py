"""Reads of large fields into numpy arrays, exact: sizes around the threshold of
the threaded copy (3 MiB) and around its 1 MiB chunks, from one thread and from
several at once (a second reader takes the plain copy), and with a world per
read (the copy's buffers outlive the worlds that read through them)."""

import gc
import threading
import time

import numpy as np
import pytest

import mumaxplus as mp

pytestmark = pytest.mark.gpu


def _magnet(nx, ny, seed):
    world = mp.World((2e-9, 2e-9, 2e-9))
    mag = mp.Ferromagnet(world, mp.Grid((nx, ny, 1)))
    mag.enable_demag = False
    m = np.random.default_rng(seed).normal(size=(3, 1, ny, nx)).astype(np.float32)
    mag.magnetization = m
    d = m.astype(np.float64)
    return world, mag, (d / np.sqrt((d * d).sum(axis=0))).astype(np.float32)


# 12 nx ny bytes: 3 MiB at 512 x 512, one chunk more at 512 x 683 (4 MiB and a row)
@pytest.mark.parametrize("size", [(511, 512), (512, 512), (513, 512), (512, 683), (1021, 1019), (1024, 1024)])
def test_exact(size):
    world, mag, want = _magnet(*size, seed=size[0])
    assert np.abs(mag.magnetization.get() - want).max() <= 6e-8  # the last bit of the host's normalisation
    got = mag.magnetization.get()
    mag.magnetization = got
    assert np.array_equal(mag.magnetization.get(), mag.magnetization.eval())


def test_several_readers():
    made = [_magnet(1024, 512 + 64 * i, seed=i) for i in range(4)]
    first = [mag.magnetization.get() for _, mag, _ in made]
    bad = []

    def read(i):
        for _ in range(10):
            if not np.array_equal(made[i][1].magnetization.get(), first[i]):
                bad.append(i)

    threads = [threading.Thread(target=read, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    for i, (_, _, want) in enumerate(made):
        assert np.abs(first[i] - want).max() <= 6e-8


def _point(n):
    """One world that reads its state once and goes: seconds of the read and the release, and the state."""
    world = mp.World((2e-9, 2e-9, 2e-9))
    mag = mp.Ferromagnet(world, mp.Grid((n, n, 1)))
    mag.enable_demag = False
    mag.magnetization = (0.0, 0.6, 0.8)
    gc.collect()
    t = time.perf_counter()
    m = mag.magnetization.get()
    del mag, world
    gc.collect()
    return time.perf_counter() - t, m


def test_a_world_per_read():
    gc.collect()
    sizes = (500, 512)  # on either side of the threaded copy's threshold
    for n in sizes:
        for _ in range(12):  # past the reads that go without the buffers
            _point(n)
    took = {n: [] for n in sizes}
    for _ in range(15):
        for n in sizes:
            s, m = _point(n)
            assert np.array_equal(m[1], np.full((1, n, n), np.float32(0.6)))
            took[n].append(s)
    # 2.9 against 3.1 ms for the read and the release; with buffers made and
    # freed for each of the larger reads 7.9 against 5.2
    assert sorted(took[512])[7] < 1.25 * sorted(took[500])[7]
