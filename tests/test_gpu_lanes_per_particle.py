"""Small systems: several lanes share a particle's stencil rows (the default
launch shape below a particle count).  Pair sums are integers, so the
trajectory equals the one-lane form's bit for bit; sizes at the edges of the
64-slot work items and of the rule (3 and 8 items per compute unit)."""
import numpy as np
import pytest

from readdygpu_amd import Simulation, workloads
from tests.test_gpu_parity import dense_spec, rich_spec

pytestmark = pytest.mark.gpu

CU = 256


def trajectories(make, steps=6, **kw):
    out = []
    for launch in ({}, {"block": 128}):          # the default shape; one lane per particle
        spec, xyz, types = make()
        with Simulation(spec, xyz, types, **kw) as sim:
            sim.set_launch_config(**launch)
            sim.simulate(steps)
            assert sim.check_invariants() == 0
            out.append(sim.copy_pos_from_device()[0])
    return out


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000, 3 * 64 * CU - 1, 3 * 64 * CU, 3 * 64 * CU + 1, 8 * 64 * CU,
                               8 * 64 * CU + 1])
def test_plain_sizes(n):
    a, b = trajectories(lambda: workloads.plain_1m(n=n, box=max(30.0, 1000.0 * (n / 1e6) ** (1 / 3)), seed=n))
    assert np.array_equal(a, b)


@pytest.mark.parametrize("make", [rich_spec, dense_spec, lambda: dense_spec(n=14000),
                                  lambda: rich_spec(cell=3.1),          # two-cell stencil
                                  lambda: rich_spec(cell=14.0),         # two cells per axis
                                  lambda: workloads.bonded_chains(500, 8, box=60.0)],
                         ids=["rich", "dense", "denser", "two_cell_stencil", "tiny_lattice", "chains"])
def test_models(make):
    a, b = trajectories(make)
    assert np.array_equal(a, b)


def test_replicas():
    spec, boxes, counts, xyz, types = workloads.batched_replicas(9, seed=4, nmin=1, nmax=4000)
    a, b = trajectories(lambda: (spec, xyz, types), replicas=(boxes, counts))
    assert np.array_equal(a, b)
