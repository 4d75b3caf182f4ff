"""The exact pass over the slots of some types, bit for bit against the
evaluation at given points: all axes +z (the packed table, four pieces at a
time) and with one tilted piece among them (the general form)."""
import numpy as np
import pytest

from readdygpu_amd import Simulation, workloads
from tests.test_gpu_composite_grid import BOX, slab, tilted

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tilt", [False, True])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8, 63, 257, 2048])
def test_types(n, tilt):
    rng = np.random.default_rng(n)
    pieces = slab(rng, n)
    if tilt:
        pieces[n // 2] = tilted(rng, 1)[0]
    spec, xyz, types = workloads.plain_10k(n=700)
    spec.box_hi = BOX
    xyz = workloads.uniform_positions(rng, 700, (0.0, 0.0, 0.0), BOX).astype(np.float32)
    with Simulation(spec, xyz, types) as sim:
        plain, _ = sim.gradients()
        sim.set_composite(pieces)
        at, _ = sim.composite_eval(xyz)
        sim.set_composite(pieces, types=[1])
        part, _ = sim.gradients()
    assert np.array_equal(part, np.where((types == 1)[:, None], plain + at, plain))
