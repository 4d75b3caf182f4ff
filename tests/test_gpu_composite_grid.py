"""The nearest-piece grid against scans over all pieces, bit for bit.

At most eight pieces are scanned, more go through the grid of candidate lists;
so the pieces are evaluated in groups of eight and the groups' results combined
by the first-argmin rule, which must equal the grid's result exactly."""
import numpy as np
import pytest

from readdygpu_amd import ATTRACTIVE, CYLINDER, DISK, OrderOnePotential, Simulation, workloads

pytestmark = pytest.mark.gpu

BOX = (150.0, 90.0, 60.0)


def piece(rng, kind, **kw):
    d = dict(k=5.0, origin=tuple(rng.uniform(-0.1, 1.1, 3) * BOX), normal=(0.0, 0.0, 1.0),
             radius=float(rng.uniform(2, 25)), height=float(rng.uniform(2, 40)) if kind == CYLINDER else 0.0)
    d.update(kw)
    return OrderOnePotential(kind, ATTRACTIVE, **d)


def slab(rng, n):
    return [piece(rng, DISK if i % 2 else CYLINDER) for i in range(n)]


def tilted(rng, n):
    return [piece(rng, DISK if i % 2 else CYLINDER, normal=tuple(rng.normal(size=3))) for i in range(n)]


def stiffnesses(rng, n):
    return [piece(rng, DISK if i % 2 else CYLINDER, k=float(rng.uniform(0.1, 20))) for i in range(n)]


def membrane(rng, n):
    out = []
    for i in range(n):
        o = rng.uniform(0, 1, 3) * BOX
        out.append(piece(rng, DISK, origin=(o[0], o[1], 24.0 if i % 3 else 36.0), radius=float(rng.uniform(3, 40))))
    return out


def duplicates(rng, n):
    few = slab(rng, 5)
    return [few[i % 5] for i in range(n)]


def wide(rng, n):
    """Cylinders that hold most of the box: energy 0 from many pieces at once."""
    return [piece(rng, CYLINDER, radius=float(rng.uniform(60, 200)), height=float(rng.uniform(30, 200))) for _ in range(n)]


def crowd(rng, n):
    """More candidates in a cell than its list holds."""
    return [piece(rng, DISK, origin=(75.0 + rng.normal() * 0.01, 45.0, 30.0 + 0.001 * i), normal=tuple(rng.normal(size=3)),
                  radius=5.0) for i in range(n)]


def points(rng, pieces):
    x = (rng.uniform(0, 1, (40_000, 3)) * BOX).astype(np.float32)
    out = (rng.uniform(-1, 2, (4000, 3)) * BOX).astype(np.float32)            # also outside the domain
    on = np.array([p.origin for p in pieces], np.float32)                     # centres and near them
    near = (np.repeat(on, 20, 0) + rng.normal(size=(20 * len(on), 3)) * 3).astype(np.float32)
    return np.concatenate([x, out, on, near])


@pytest.mark.parametrize("make", [slab, tilted, stiffnesses, membrane, duplicates, wide, crowd])
@pytest.mark.parametrize("n", [9, 33, 257, 600])
def test_grid_equals_scan(make, n):
    rng = np.random.default_rng(n)
    pieces = make(rng, n)
    x = points(rng, pieces)
    spec, xyz, types = workloads.plain_10k(n=100)
    spec.box_hi = BOX
    xyz = (xyz * np.float32(0.5)).astype(np.float32)
    with Simulation(spec, xyz, types) as sim:
        best = np.full(len(x), np.inf, np.float32)
        grad = np.zeros_like(x)
        for i in range(0, n, 8):
            sim.set_composite(pieces[i:i + 8])
            g, e = sim.composite_eval(x)
            take = e < best
            best[take] = e[take]
            grad[take] = g[take]
        sim.set_composite(pieces)
        g, e = sim.composite_eval(x)
        assert np.array_equal(e, best)
        assert np.array_equal(g, grad)
        # the step's pass, on every type and on one of two
        at, _ = sim.composite_eval(xyz)
        sim.set_composite([])
        plain, _ = sim.gradients()
        for on in ([0, 1], [1]):
            sim.set_composite(pieces, types=on)
            with_ext, _ = sim.gradients()
            assert np.array_equal(with_ext, np.where(np.isin(types, on)[:, None], plain + at, plain))


def test_domain_follows_the_boxes():
    """New boxes after the pieces were set: the lists are built again."""
    rng = np.random.default_rng(3)
    pieces = slab(rng, 100)
    x = points(rng, pieces)
    spec, xyz, types = workloads.plain_10k(n=200)
    with Simulation(spec, xyz, types) as sim:
        sim.set_composite(pieces)
        sim.simulate(2)
        a = sim.composite_eval(x)
        boxes = np.array([[-40.0, 20.0, 0.0, 60.0, 10.0, 70.0], [100.0, 160.0, 30.0, 90.0, 0.0, 60.0]])
        inside = np.concatenate([workloads.uniform_positions(rng, 100, b[0::2], b[1::2]) for b in boxes])
        sim.set_replicas(boxes, np.array([100, 100]), inside, types)
        b = sim.composite_eval(x)
        sim.simulate(2)
        c = sim.composite_eval(x)
    for u, v, w in zip(a, b, c):
        assert np.array_equal(u, v) and np.array_equal(u, w)
