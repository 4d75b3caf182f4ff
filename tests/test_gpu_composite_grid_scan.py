"""The nearest-piece grid where a wave scans all pieces: lists that overflow in
every cell, points outside the domain among points inside it, at the edges of
the staged chunk (64 pieces) and of a wave; bit for bit against evaluations of
eight pieces each."""
import numpy as np
import pytest

from readdygpu_amd import Simulation, workloads
from tests.test_gpu_composite_grid import BOX, crowd, slab
from tests.test_gpu_composite_grid_tall import scan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make", [crowd, slab])
@pytest.mark.parametrize("n", [40, 63, 64, 65, 127, 128, 129, 2048])
def test_scans(make, n):
    rng = np.random.default_rng(n)
    pieces = make(rng, n)
    spec, xyz, types = workloads.plain_10k(n=100)
    spec.box_hi = BOX
    xyz = (xyz * np.float32(0.5)).astype(np.float32)
    with Simulation(spec, xyz, types) as sim:
        for m in (1, 63, 64, 65, 5000):
            x = (rng.uniform(0, 1, (m, 3)) * BOX).astype(np.float32)
            x[::3] += np.float32([0, 0, 1.5 * BOX[2]])
            x[m // 2] = np.float32(BOX)                  # the domain's upper corner
            grad, best = scan(sim, pieces, x)
            sim.set_composite(pieces)
            for _ in range(5):                           # before and after the lists are built
                g, e = sim.composite_eval(x)
                assert np.array_equal(e, best) and np.array_equal(g, grad), m
        # the step's pass, particles that do not fill the last wave
        at, _ = sim.composite_eval(xyz)
        sim.set_composite([])
        plain, _ = sim.gradients()
        sim.set_composite(pieces)
        sim.simulate(0)
        with_ext, _ = sim.gradients()
        assert np.array_equal(with_ext, plain + at)


def test_data_wider_than_the_boxes():
    """Samples of which most lie outside the boxes: the training set's scale and
    the validation error equal those of a handle whose boxes hold all of them."""
    rng = np.random.default_rng(2)
    pieces = slab(rng, 100)
    out = []
    for hi in (BOX, tuple(3.0 * v for v in BOX)):
        spec, xyz, types = workloads.plain_10k(n=100)
        spec.box_hi = hi
        with Simulation(spec, (xyz * np.float32(0.5)).astype(np.float32), types) as sim:
            sim.set_composite(pieces)
            sim.surrogate_init(3)
            sim.set_surrogate_norm((0, 0, 0), tuple(2.5 * v for v in BOX), 1.0)
            for _ in range(5):                       # before and after the lists are built
                r = [sim.surrogate_make_data(70_001, seed=4), sim.surrogate_validate(10_001, seed=5)]
                out.append(r)
    assert all(r == out[0] for r in out), out
