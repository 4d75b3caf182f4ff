"""The nearest-piece composite before and after its grid is built (it takes a few
passes over the same pieces): the same bits from every pass, at given points and
on the particles' slots, and a run's steps do not depend on when that is."""
import numpy as np
import pytest

from readdygpu_amd import Simulation, workloads
from tests import test_gpu_composite_grid as shapes
from tests.test_gpu_composite_grid_tall import scan

pytestmark = pytest.mark.gpu

BOX = shapes.BOX
MAKERS = [shapes.slab, shapes.tilted, shapes.stiffnesses, shapes.membrane, shapes.duplicates, shapes.wide, shapes.crowd]


def system(n=1000):
    spec, xyz, types = workloads.plain_10k(n=n)
    spec.box_hi = BOX
    rng = np.random.default_rng(n)
    return spec, workloads.uniform_positions(rng, n, (0, 0, 0), BOX), types


@pytest.mark.parametrize("make", MAKERS)
@pytest.mark.parametrize("n", [9, 12, 33, 257, 600])
def test_points_and_slots(make, n):
    rng = np.random.default_rng(n)
    pieces = make(rng, n)
    x = shapes.points(rng, pieces)
    spec, xyz, types = system()
    with Simulation(spec, xyz, types) as sim:
        grad, best = scan(sim, pieces, x)
        sim.set_composite([])
        plain, _ = sim.gradients()
        at, _ = scan(sim, pieces, xyz)
        sim.set_composite(pieces)
        for _ in range(5):
            g, e = sim.composite_eval(x)
            assert np.array_equal(e, best) and np.array_equal(g, grad)
        sim.set_composite(pieces)
        for _ in range(5):
            assert np.array_equal(sim.gradients()[0], plain + at)


@pytest.mark.parametrize("frames", [(40,), (1,) * 10, (0, 3, 7), (2, 2, 16, 20)])
def test_steps(frames):
    pieces = shapes.slab(np.random.default_rng(1), 100)
    spec, xyz, types = system()
    spec.dt = 0.002
    out = []
    for plan in (frames, (sum(frames),)):
        with Simulation(spec, xyz, types) as sim:
            sim.set_composite(pieces)
            for k in plan:
                sim.simulate(k)
            out.append(sim.copy_pos_from_device()[0].copy())
    assert np.array_equal(out[0], out[1])
