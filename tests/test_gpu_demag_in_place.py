"""The demag operator with its result written over its source, on the GPU.

The field must be that of the source as it was at the call, also where a small
grid's field is otherwise summed directly in one launch: m overwritten by h,
shifted arrays that overlap in part, and the per-cell Ms array overwritten,
through both entry points, against the field written to an array of its own.
"""

import numpy as np
import pytest

from helpers import DeviceBuffer, random_unit

import mumaxplus as mp

pytestmark = pytest.mark.gpu

CS = (2e-9, 2.5e-9, 3e-9)


@pytest.mark.parametrize("entry", ["exec", "exec_noalloc"])
@pytest.mark.parametrize("size", [(64, 64, 1), (33, 9, 4), (41, 16, 1), (33, 17, 1), (40, 24, 6), (20, 12, 9)])
def test_field_over_its_source(size, entry):
    nx, ny, nz = size
    n = nx * ny * nz
    rng = np.random.default_rng(n)
    m = random_unit(rng, (nz, ny, nx)).astype(np.float32)
    plan = mp._cpp.DemagPlan(size, CS)
    run = getattr(plan, entry)
    md, hd = DeviceBuffer.from_host(m), DeviceBuffer(m.nbytes)
    run(md.ptr, hd.ptr, msat_uniform=8e5)
    want = hd.to_host(np.float32, m.shape)
    scale = np.abs(want).max()
    assert scale > 0
    # the direct sum and the passes round differently: 4e-7 of the largest field
    # each against 64 bits
    tol = 8e-7 * scale
    run(md.ptr, md.ptr, msat_uniform=8e5)
    assert np.abs(md.to_host(np.float32, m.shape) - want).max() <= tol
    # two thirds of h over the source: floats n .. 4n of a buffer of 4n
    both = DeviceBuffer.from_host(np.concatenate([m.ravel(), np.zeros(n, np.float32)]))
    run(both.ptr, both.ptr + 4 * n, msat_uniform=8e5)
    assert np.abs(both.to_host(np.float32, (4, n))[1:].reshape(m.shape) - want).max() <= tol
    # the last component over the per-cell Ms
    msat = np.full(n, 8e5, np.float32)
    md2 = DeviceBuffer.from_host(m)
    hs = DeviceBuffer.from_host(np.concatenate([np.zeros(2 * n, np.float32), msat]))
    run(md2.ptr, hs.ptr, msat_ptr=hs.ptr + 8 * n)
    assert np.abs(hs.to_host(np.float32, m.shape) - want).max() <= tol
