"""Points and results through the same pinned buffer: calls on both sides of the
size up to which the results lie behind the points (64 KB: 2,340 points of the
composite, 2,730 of the network), of the pinned memory's end (4 MB) and in turn,
against one call of all points."""
import numpy as np
import pytest

from readdygpu_amd import Simulation, workloads

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 2340, 2341, 2730, 2731, 5461, 5462, 262_144, 262_145, 349_525, 349_526]


def test_sizes_in_turn():
    spec, pieces, xyz, types = workloads.learned_slab(n=500, n_pieces=20)
    rng = np.random.default_rng(1)
    x = workloads.uniform_positions(rng, max(SIZES), spec.box_lo, spec.box_hi).astype(np.float32)
    xn = rng.uniform(-1, 1, (max(SIZES), 3)).astype(np.float32)
    with Simulation(spec, xyz, types) as sim:
        sim.set_composite(pieces)
        sim.surrogate_init(2)
        grad, energy = sim.composite_eval(x)
        y = sim.surrogate_predict(xn)
        for m in SIZES + SIZES[::-1]:
            first = int(rng.integers(0, max(SIZES) - m + 1))
            g, e = sim.composite_eval(x[first:first + m])
            assert np.array_equal(g, grad[first:first + m]) and np.array_equal(e, energy[first:first + m]), m
            assert np.array_equal(sim.surrogate_predict(xn[first:first + m]), y[first:first + m]), m
