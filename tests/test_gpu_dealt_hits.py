"""Crowded systems: a wave's hits go to one queue and are dealt to its lanes
(the default launch shape where a particle expects enough partners, past the
sizes at which lanes share a particle).  Pair sums are integers, so the
trajectory equals the other one-lane form's bit for bit: partly filled and
single-particle waves, the smallest lattices, waves whose hits overflow the
queue, both sides of the rule, bonds, external potentials."""
import numpy as np
import pytest

from readdygpu_amd import Simulation, workloads

pytestmark = pytest.mark.gpu

CU = 256
WAVES = 8 * CU + 1                  # fewer 64-slot items: several lanes per particle


def trajectories(spec, xyz, types, steps=5, **kw):
    out = []
    for launch in ({}, {"block": 128}):          # the default shape; each lane its own list
        with Simulation(spec, xyz, types, **kw) as sim:
            sim.set_launch_config(**launch)
            sim.simulate(steps)
            assert sim.check_invariants() == 0
            out.append(sim.copy_pos_from_device()[0])
    return out


def boxes(cells, nmin, nmax, clump=1.0, seed=5):
    """WAVES or more boxes of `cells` cells per axis, the particles in the
    leading `clump` of each axis."""
    spec = workloads.batched_replicas(1, nmin=1, nmax=2)[0]
    spec.dt = 0.02
    cell = 1.01 * 2.0 * max(t.radius for t in spec.types)
    edge = 1.001 * cell * np.asarray(cells, float)
    rng = np.random.default_rng(seed)
    counts, items = [], 0
    while items < WAVES:
        counts.append(int(rng.integers(nmin, nmax + 1)))
        items += (counts[-1] + 63) // 64
    n = sum(counts)
    bounds = np.tile(np.stack([np.zeros(3), edge], 1).reshape(6), (len(counts), 1))
    types = rng.integers(0, 2, n).astype(np.int32)
    return spec, bounds, np.asarray(counts), rng.uniform(0, clump * edge, (n, 3)), types


@pytest.mark.parametrize("cells,nmin,nmax,clump", [
    ((3, 3, 3), 1, 1, 1.0),             # one lane per wave
    ((3, 3, 3), 1, 130, 1.0),           # partly filled waves; the densest overflow the queue
    ((3, 3, 3), 128, 129, 0.3),         # one cell holds nearly all: a row alone overflows it
    ((4, 3, 5), 60, 66, 1.0),
    ((7, 4, 3), 1, 200, 0.5),
    ((2, 3, 3), 20, 70, 1.0),           # two cells per axis: not the queue's
    ((8, 8, 8), 110, 110, 1.0),         # 5.8 candidates, 0.6 partners
    ((8, 8, 8), 80, 80, 1.0),           # 4.2 candidates: the sparse form's
], ids=str)
def test_boxes(cells, nmin, nmax, clump):
    spec, bounds, counts, xyz, types = boxes(cells, nmin, nmax, clump)
    a, b = trajectories(spec, xyz, types, replicas=(bounds, counts))
    assert np.array_equal(a, b)


@pytest.mark.parametrize("make", [lambda: workloads.plain_1m(n=64 * WAVES - 1, box=350.0),
                                  lambda: workloads.bonded_chains(17000, 8, box=190.0)],
                         ids=["external_potential", "chains"])
def test_models(make):
    a, b = trajectories(*make())
    assert np.array_equal(a, b)
