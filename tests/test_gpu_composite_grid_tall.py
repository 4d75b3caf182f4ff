"""The nearest-piece grid against scans of at most eight pieces, bit for bit,
where rounding decides the nearest piece: in a box far taller than wide the
squared distance to a disk's plane absorbs the radial part (at 1e5 from the
plane its FP32 spacing is 1,024), so that coplanar pieces tie and the one of
the lower index is the nearest."""
import numpy as np
import pytest

from readdygpu_amd import ATTRACTIVE, CYLINDER, DISK, OrderOnePotential, Simulation, workloads

pytestmark = pytest.mark.gpu


def scan(sim, pieces, x):
    """First-argmin rule over evaluations of eight pieces each."""
    best = np.full(len(x), np.inf, np.float32)
    grad = np.zeros_like(x)
    for i in range(0, len(pieces), 8):
        sim.set_composite(pieces[i:i + 8])
        g, e = sim.composite_eval(x)
        take = e < best
        best[take] = e[take]
        grad[take] = g[take]
    return grad, best


def compare(box, pieces, seed, m=60_000):
    rng = np.random.default_rng(seed)
    x = (rng.uniform(0, 1, (m, 3)) * box).astype(np.float32)
    spec, xyz, types = workloads.plain_10k(n=100)
    spec.box_hi = box
    with Simulation(spec, (xyz * np.float32(0.2)).astype(np.float32), types) as sim:
        grad, best = scan(sim, pieces, x)
        sim.set_composite(pieces)
        for _ in range(5):                     # before and after the lists are built
            g, e = sim.composite_eval(x)
            assert np.array_equal(e, best)
            assert np.array_equal(g, grad)


@pytest.mark.parametrize("height", [1e3, 1e4, 3e4, 4e4, 5e4, 7e4, 1e5, 1e6])
@pytest.mark.parametrize("n,planes,kind", [(24, 1, DISK), (48, 2, DISK), (24, 1, CYLINDER), (600, 1, DISK)])
def test_tall_boxes(height, n, planes, kind):
    """24 pieces of a plane fit a cell's list."""
    box = (20.0, 20.0, height)
    rng = np.random.default_rng(int(height) + planes)
    pieces = []
    for i in range(n):
        z = (0.0, 1.0)[i % planes] * height
        pieces.append(OrderOnePotential(kind, ATTRACTIVE, k=5.0, origin=(*rng.uniform(0, 20, 2), z), normal=(0.0, 0.0, 1.0),
                                        radius=float(rng.uniform(0.05, 0.5)), height=2.0 if kind == CYLINDER else 0.0))
    compare(box, pieces, planes)
