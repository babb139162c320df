"""The one-thread-both-sublattices kernel of uniform antiferromagnets and the
elastic kernels of periodic films, against the FP64 oracle: a step of the
coupled equations at the sizes where the rules can go wrong (rows that are no
multiple of a block, one to three cells along an axis, layers, open, periodic
and partly periodic axes, every switchable term)."""

import numpy as np
import pytest

from helpers import random_unit
from oracle import model as omodel

import mumaxplus as mp

pytestmark = pytest.mark.gpu

CS = (2e-9, 2.5e-9, 3e-9)
OPEN, FILM = (0, 0, 0), (1, 1, 0)
CASES = [((65, 5, 1), FILM, True), ((3, 3, 1), FILM, True), ((70, 4, 1), OPEN, True), ((64, 8, 1), (1, 0, 0), True),
         ((5, 1, 1), OPEN, False), ((9, 7, 3), OPEN, True), ((6, 5, 4), (1, 1, 1), True), ((130, 3, 2), FILM, False),
         ((2, 2, 1), FILM, True), ((2, 2, 512), OPEN, False), ((4, 2, 513), OPEN, False), ((3, 3, 513), OPEN, False)]


@pytest.mark.parametrize("nn", [0.0, -3e-12])
@pytest.mark.parametrize("size,per,elastic", CASES)
def test_one_step(size, per, elastic, nn):
    rng = np.random.default_rng(sum(size) + int(elastic))
    box = tuple(n if p else 0 for n, p in zip(size, per))
    world = mp.World(CS, mastergrid=mp.Grid(box), pbc_repetitions=per)
    afm = mp.Antiferromagnet(world, mp.Grid(size))
    ow = omodel.World(CS, mastergrid=box, pbc=per)
    oa = ow.add_antiferromagnet(size, defer_timestep=True)
    sub = {"msat": 566e3, "aex": 2.48e-12, "alpha": 0.1, "ku1": 2e5, "anisU": (0.2, 0.3, 1.0)}
    for k, v in sub.items():
        setattr(afm, k, v)
        for s in (oa.sub1, oa.sub2):
            s.set(k, v)
    host = {"afmex_cell": -4e-12, "afmex_nn": nn}
    for k, v in host.items():
        setattr(afm, k, v)
        oa.set(k, v)
    afm.dmi_tensors.set_bulk_dmi(1e-3)
    for t in (oa, oa.sub1, oa.sub2):
        t.set("xyz", 1e-3)
        t.set("yxz", -1e-3)
        t.set("zxy", 1e-3)
    world.bias_magnetic_field = (0.02, -0.01, 0.03)
    ow.bias = (0.02, -0.01, 0.03)
    shape = size[::-1]
    m1, m2 = random_unit(rng, shape).astype(np.float32), random_unit(rng, shape).astype(np.float32)
    afm.sub1.magnetization, afm.sub2.magnetization = m1, m2
    oa.sub1.set_m(afm.sub1.magnetization.get().astype(float))
    oa.sub2.set_m(afm.sub2.magnetization.get().astype(float))
    if elastic:
        el = {"C11": 283e9, "C12": 166e9, "C44": 58e9, "rho": 8900.0, "eta": 1e12}
        afm.B1 = afm.B2 = -8.8e6
        for s in (oa.sub1, oa.sub2):
            s.set("B1", -8.8e6)
            s.set("B2", -8.8e6)
        afm.enable_elastodynamics = True
        oa.enable_elastodynamics = True
        for k, v in el.items():
            setattr(afm, k, v)
            oa.set(k, v)
        u = (1e-12 * rng.normal(size=(3,) + shape)).astype(np.float32)
        afm.elastic_displacement = u
        oa.u = u.astype(float)
    world.timesolver.set_method("DormandPrince")
    ow.solver.set_method("DormandPrince", defer_timestep=True)
    world.timesolver.adaptive_timestep, world.timesolver.timestep = False, 2e-15
    ow.solver.adaptive, ow.solver.dt = False, 2e-15
    start = [s.m.copy() for s in (oa.sub1, oa.sub2)]
    world.timesolver.steps(2)
    ow.solver.steps(2)
    for g, o, m0 in ((afm.sub1, oa.sub1, start[0]), (afm.sub2, oa.sub2, start[1])):
        dm, want = g.magnetization.get() - m0, o.m - m0
        # the move of two steps, in FP32 m (2^-24 each) and fields of 1e-5
        assert np.abs(dm - want).max() <= 2e-5 * np.abs(want).max() + 2e-7
    if elastic:
        for got, want in ((afm.elastic_displacement.get(), oa.u), (afm.elastic_velocity.get(), oa.v)):
            assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max()


# Every parameter different on the two sublattices, and the inter-sublattice
# tensor different from both of theirs.
SUBS = ({"msat": 566e3, "aex": 2.48e-12, "alpha": 0.1, "ku1": 2e5, "ku2": 3e5, "anisU": (0.2, 0.3, 1.0), "B1": -8.8e6,
         "B2": -1e6},
        {"msat": 812e3, "aex": 4.1e-12, "alpha": 0.23, "ku1": -3e5, "ku2": 1e5, "anisU": (1.0, -0.4, 0.1), "B1": -1e6,
         "B2": -1.1e7})
TENSORS = ({"xyz": 1e-3, "yxz": -0.7e-3, "zxy": 1.3e-3, "xxz": 0.4e-3, "yyz": 0.9e-3},
           {"xyz": -0.5e-3, "yxz": 0.8e-3, "zxy": 0.6e-3, "xxy": 1.1e-3, "zyz": -1.2e-3},
           {"xyz": 0.7e-3, "yxz": 1.2e-3, "zxy": -0.4e-3, "yxy": 0.5e-3, "zxz": 0.3e-3})


def own_sublattices(size, per, strain, nn=-3e-12, subs=SUBS, tensors=TENSORS):
    """(host parameters, per-sublattice parameters, tensors, m, strain settings) of one case, for both models."""
    rng = np.random.default_rng(sum(size))
    shape = size[::-1]
    host = {"afmex_cell": -4e-12, "afmex_nn": nn}
    el = {"C11": 283e9, "C12": 166e9, "C44": 58e9, "rho": 8900.0, "eta": 1e12} if strain == "elastic" else {}
    if strain == "rigid":
        el = {"rigid_norm_strain": (4e-3, -6e-3, 2e-3), "rigid_shear_strain": (-3e-3, 5e-3, 7e-3)}
    m = [random_unit(rng, shape).astype(np.float32) for _ in range(2)]
    u = (4e-12 * rng.normal(size=(3,) + shape)).astype(np.float32)
    return host, subs, tensors, m, el, u


def oracle_move(size, per, case, strain, start):
    """The move of two steps of the FP64 model from `start`."""
    host, subs, tensors, _, el, u = case
    box = tuple(n if p else 0 for n, p in zip(size, per))
    ow = omodel.World(CS, mastergrid=box, pbc=per)
    oa = ow.add_antiferromagnet(size, defer_timestep=True)
    for s, params, tensor in zip((oa.sub1, oa.sub2), subs, tensors):
        for k, v in {**params, **tensor}.items():
            s.set(k, v)
    for k, v in {**host, **tensors[2]}.items():
        oa.set(k, v)
    ow.bias = (0.02, -0.01, 0.03)
    if strain == "elastic":
        oa.enable_elastodynamics = True
        oa.u = u.astype(float)
    for k, v in el.items():
        oa.set(k, v)
    for s, m in zip((oa.sub1, oa.sub2), start):
        s.set_m(m.astype(float))
    ow.solver.set_method("DormandPrince", defer_timestep=True)
    ow.solver.adaptive, ow.solver.dt = False, 2e-15
    ow.solver.steps(2)
    return [s.m - m for s, m in zip((oa.sub1, oa.sub2), start)]


def bound(want):
    # FP32 m (2^-24 each step and once more in the difference) and fields of 1e-5
    return 2e-5 * np.abs(want).max() + 2e-7


@pytest.mark.parametrize("strain", ["none", "elastic", "rigid"])
@pytest.mark.parametrize("size,per", [((9, 7, 3), OPEN), ((70, 4, 1), OPEN), ((65, 5, 1), FILM), ((6, 5, 4), (1, 1, 1)),
                                      ((5, 1, 1), OPEN)])
def test_sublattices_of_their_own(size, per, strain):
    case = own_sublattices(size, per, strain)
    host, subs, tensors, m, el, u = case
    box = tuple(n if p else 0 for n, p in zip(size, per))
    world = mp.World(CS, mastergrid=mp.Grid(box), pbc_repetitions=per)
    afm = mp.Antiferromagnet(world, mp.Grid(size))
    for s, params, tensor, m0 in zip((afm.sub1, afm.sub2), subs, tensors, m):
        for k, v in params.items():
            setattr(s, k, v)
        for k, v in tensor.items():
            setattr(s.dmi_tensor, k, v)
        s.magnetization = m0
    for k, v in host.items():
        setattr(afm, k, v)
    for k, v in tensors[2].items():
        setattr(afm.dmi_tensor, k, v)
    world.bias_magnetic_field = (0.02, -0.01, 0.03)
    if strain == "elastic":
        afm.enable_elastodynamics = True
        afm.elastic_displacement = u
    for k, v in el.items():
        setattr(afm, k, v)
    start = [s.magnetization.get() for s in (afm.sub1, afm.sub2)]
    world.timesolver.set_method("DormandPrince")
    world.timesolver.adaptive_timestep, world.timesolver.timestep = False, 2e-15
    world.timesolver.steps(2)
    for s, m0, want in zip((afm.sub1, afm.sub2), start, oracle_move(size, per, case, strain, start)):
        assert np.abs(s.magnetization.get() - m0 - want).max() <= bound(want)
