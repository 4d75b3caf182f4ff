"""Sparse systems: a particle's candidates are listed before they are tested
(the default launch shape below five candidates a particle, past the sizes at
which lanes share a particle).  Pair sums are integers, so the trajectory
equals the walk by rows' bit for bit: single particles, the smallest lattices,
lists at and past their 12 entries, runs of more than four, homes at the x
edge, bonds, external potentials, both sides of the rule."""
import numpy as np
import pytest

from readdygpu_amd import workloads
from tests.test_gpu_dealt_hits import WAVES, boxes, trajectories

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,nmin,nmax,clump", [
    ((3, 3, 3), 1, 2, 1.0),
    ((3, 3, 3), 4, 5, 1.0),
    ((5, 5, 5), 20, 23, 1.0),
    ((12, 12, 12), 1, 130, 1.0),        # partly filled waves
    ((8, 8, 8), 90, 90, 1.0),           # 4.7 candidates
    ((8, 8, 8), 96, 96, 1.0),           # 5.1: past the rule
    ((12, 12, 12), 200, 300, 0.25),     # every list overflows
    ((12, 12, 12), 40, 64, 0.45),       # lists about full
    ((12, 12, 12), 3, 6, 0.08),         # all in one cell: runs of 3 to 6
    ((40, 3, 3), 60, 66, 1.0),
    ((2, 9, 9), 20, 30, 1.0),           # two cells on an axis: not listed
], ids=str)
def test_boxes(cells, nmin, nmax, clump):
    spec, bounds, counts, xyz, types = boxes(cells, nmin, nmax, clump)
    a, b = trajectories(spec, xyz, types, replicas=(bounds, counts))
    assert np.array_equal(a, b)


@pytest.mark.parametrize("make", [lambda: workloads.plain_1m(n=64 * WAVES - 1, box=600.0),
                                  lambda: workloads.bonded_chains(17000, 8, box=900.0)],
                         ids=["external_potential", "chains"])
def test_models(make):
    a, b = trajectories(*make())
    assert np.array_equal(a, b)
