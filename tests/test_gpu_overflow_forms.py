"""A pair term beyond the fixed-point range is reported by every form of the
force kernel and by both gradient kernels, also where the lane that evaluates
it holds no particle (hits dealt to the lanes of a wave).  Which kernel each
system runs is checked without a GPU."""
import ctypes

import numpy as np
import pytest

from readdygpu_amd import HARMONIC, REPULSIVE, OrderTwoPotential, ParticleType, RdError, Simulation, SystemSpec
from tests.test_gpu_dealt_hits import boxes, trajectories

pytestmark = pytest.mark.gpu

CU = 256
R0 = 2.0                             # range of the pair term
K = 3.5e8                            # k (r0 - r): 7e8 at contact, 3.5e7 at 0.95 r0 (the range is 5e8)


def system(form, offend):
    """Boxes of one wave each; in the last one particles 0 and 1 lie 0.02 apart
    if `offend`.  The other particles of a box lie 0.95 r0 or more from each
    other and from these."""
    boxes, cells, cell = {"lanes9": (10, 3, 1.01), "lanes3": (3 * CU + 5, 3, 1.01), "sparse": (8 * CU + 5, 3, 1.01),
                          "rows": (8 * CU + 5, 3, 2.1), "dealt": (8 * CU + 5, 3, 1.01),
                          "dealt_idle_lane": (8 * CU + 5, 3, 1.01)}[form]
    per = 2 if form == "sparse" else 6
    c = cell * R0
    edge = cells * c * 1.0001
    spec = SystemSpec(box_lo=(0, 0, 0), box_hi=(edge,) * 3, dt=1e-13, seed=3, cell_size=c)
    spec.types = [ParticleType("A", 1.0, R0 / 2)]
    spec.pot2 = [OrderTwoPotential(HARMONIC, REPULSIVE, K)]
    # 0 and 1 in the middle cell; with hits dealt to the lanes the first eight
    # entries of the queue are theirs with 2 .. 5 in the layer below, and lanes
    # 6 and up hold no particle
    mid = np.array([0.5, 0.5, 0.5]) * edge
    x = np.empty((6, 3))
    x[0] = mid + (0, 0, -0.3 * c)
    x[1] = x[0] + (0.02, 0, 0)
    near = 0.95 * R0 if form == "dealt_idle_lane" else 1.2 * R0
    for i, d in enumerate([(1, 0), (-1, 0), (0, 1), (0, -1)]):
        down = 0.35 * c
        x[2 + i] = x[0] + (0.01 + d[0] * np.sqrt(near ** 2 - down ** 2), d[1] * np.sqrt(near ** 2 - down ** 2), -down)
    x = x[:per]
    xyz = np.tile(x, (boxes, 1)).astype(np.float32)
    apart = np.arange(1, len(xyz), per)                 # particle 1 of each box, away from 0
    xyz[apart, 2] += np.float32(1.3 * R0)
    if offend:
        xyz[apart[-1]] = x[1]
    bounds = np.tile(np.array([0.0, edge] * 3), (boxes, 1))
    return spec, xyz, np.zeros(len(xyz), np.int32), (bounds, np.full(boxes, per))


FORMS = ["lanes9", "lanes3", "sparse", "rows", "dealt", "dealt_idle_lane"]


@pytest.mark.parametrize("form", FORMS)
def test_steps(form):
    spec, xyz, types, replicas = system(form, False)
    with Simulation(spec, xyz, types, replicas=replicas) as sim:
        sim.simulate(2)
    spec, xyz, types, replicas = system(form, True)
    for shape in ({}, {"block": 128}, {"ppt": 2}, {"kernel": 2}):
        with Simulation(spec, xyz, types, replicas=replicas) as sim:
            sim.set_launch_config(**shape)
            with pytest.raises(RdError, match="fixed-point range"):
                sim.simulate(1)


@pytest.mark.parametrize("form", ["lanes9", "lanes3", "dealt"])
def test_gradients(form):
    for offend in (False, True):
        spec, xyz, types, replicas = system(form, offend)
        with Simulation(spec, xyz, types, replicas=replicas) as sim:
            if not offend:
                sim.gradients()
                continue
            with pytest.raises(RdError, match="fixed-point range"):
                sim.gradients()


@pytest.mark.parametrize("n", [65, 129])
def test_dealt_single_particle_waves(n):
    """The last wave of every box holds one particle."""
    spec, bounds, counts, xyz, types = boxes((3, 3, 3), n, n)
    a, b = trajectories(spec, xyz, types, replicas=(bounds, counts))
    assert np.array_equal(a, b)


def test_compute_units():
    """The sizes here and in the other tests of the launch rules are for 256."""
    spec, xyz, types, replicas = system("lanes9", False)
    with Simulation(spec, xyz, types, replicas=replicas) as sim:
        name = ctypes.create_string_buffer(256)
        assert sim.lib.rd_device_name(0, name, 256) == 0
        assert name.value.decode().endswith(" %dCU" % CU)
