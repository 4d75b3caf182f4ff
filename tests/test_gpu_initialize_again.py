"""A second rd_initialize: what goes up are the positions and types that were
last set or last copied out, or those that reactions left; the steps after it
follow from them.  Sizes on both sides of the pinned copy (262,144 particles)
and of the gradient kernels' line; calls in between that use device scratch."""
import numpy as np
import pytest

from readdygpu_amd import Simulation, workloads

pytestmark = pytest.mark.gpu

SIZES = [1, 65, 2000, 60_000, 262_145]


def make(n):
    return workloads.plain_1m(n=n, box=max(30.0, 1000.0 * (n / 1e6) ** (1 / 3)), seed=n)


def state(sim):
    x, t = sim.copy_pos_from_device()
    return x.copy(), t.copy()


def same(a, b):
    return np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("n", SIZES)
def test_copied_positions_go_up(n):
    spec, xyz, types = make(n)
    with Simulation(spec, xyz, types) as sim:
        sim.simulate(5)
        a = state(sim)
        assert not np.array_equal(a[0], xyz)
        sim.initialize()
        assert same(state(sim), a) and sim.info().step == 5
        sim.initialize()
        assert same(state(sim), a)
        sim.simulate(3)                       # the run goes on as one without the calls
        b = state(sim)
        assert sim.check_invariants() == 0
    with Simulation(spec, xyz, types) as sim:
        sim.simulate(8)
        assert same(state(sim), b)


@pytest.mark.parametrize("n", SIZES)
def test_last_copied_not_current(n):
    """Steps after the copy are dropped, as where the host holds the arrays;
    the calls between use the device's scratch."""
    spec, xyz, types = make(n)
    with Simulation(spec, xyz, types) as sim:
        sim.simulate(4)
        a = state(sim)
        sim.simulate(4)
        sim.gradients()
        sim.cell_ids()
        sim.neighbor_pairs()
        sim.frame_copy()
        sim.simulate(2)
        sim.frame_rewind()
        sim.initialize()
        assert same(state(sim), a)
        assert sim.check_invariants() == 0


@pytest.mark.parametrize("n", SIZES)
def test_set_positions_go_up(n):
    spec, xyz, types = make(n)
    with Simulation(spec, xyz, types) as sim:
        sim.simulate(3)
        sim.initialize()
        assert same(state(sim), (xyz, types))


@pytest.mark.parametrize("copy", [False, True])
@pytest.mark.parametrize("n", [65, 2000, 262_145])
def test_reactions_go_up(n, copy):
    """The box lies away from the origin: a position left at zero is outside."""
    spec, xyz, types = make(n)
    shift = np.float32(100.0)
    spec.box_lo = tuple(v + 100.0 for v in spec.box_lo)
    spec.box_hi = tuple(v + 100.0 for v in spec.box_hi)
    for p in spec.pot1:
        p.origin = tuple(v + 100.0 for v in p.origin)
    with Simulation(spec, xyz + shift, types) as sim:
        sim.simulate(2)
        x, t = state(sim)
        rows = [[0, 1 - t[0], *x[0], 0], [1, -1, *x[1], 1], [-1, 1, *x[2], -1], [-1, 0, *x[3], -1]]
        sim.apply_reactions(np.concatenate([[len(rows)], np.asarray(rows, np.float32).reshape(-1)]).astype(np.float32))
        ref = np.concatenate([x[2:], x[:1], x[2:4]]), np.concatenate([t[2:], [1 - t[0], 1, 0]]).astype(np.int32)
        if copy:
            assert same(state(sim), ref)
        sim.initialize()
        assert same(state(sim), ref)
        assert sim.check_invariants() == 0
        sim.simulate(2)


def test_replicas():
    spec, boxes, counts, xyz, types = workloads.batched_replicas(5, seed=4, nmin=1, nmax=4000)
    with Simulation(spec, xyz, types, replicas=(boxes, counts)) as sim:
        sim.simulate(3)
        a = state(sim)
        sim.simulate(3)
        sim.gradients()
        sim.initialize()
        assert same(state(sim), a)
        assert sim.check_invariants() == 0
