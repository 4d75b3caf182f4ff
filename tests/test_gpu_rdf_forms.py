"""RDF counts of every launch form (16, 4 and 2 lanes per particle) against the
oracle, bit for bit: sizes on both sides of the rule's lines (2 and 16 work
items of 64 particles per compute unit), boxes with an offset, a partial top
cell and unequal edges, ranges that are no multiple of the cell, replicas that
share a workgroup, and distances that fall exactly on bin edges."""
import numpy as np
import pytest

from oracle import oracle as orc
from readdygpu_amd import HARMONIC, REPULSIVE, OrderTwoPotential, ParticleType, Simulation, SystemSpec, workloads

pytestmark = pytest.mark.gpu

CU = 256


def make(n, lo, hi, cell, seed):
    spec = SystemSpec(box_lo=lo, box_hi=hi, dt=0.01, seed=seed, cell_size=cell)
    spec.types = [ParticleType("A", 1.0, 1.0), ParticleType("B", 0.5, 1.5), ParticleType("C", 2.0, 0.8)]
    spec.pot2 = [OrderTwoPotential(HARMONIC, REPULSIVE, 10.0)]
    rng = np.random.default_rng(seed)
    return spec, workloads.uniform_positions(rng, n, lo, hi), rng.integers(0, 3, n).astype(np.int32)


@pytest.mark.parametrize("n", [1, 64, 65, 2 * 64 * CU, 2 * 64 * CU + 1, 16 * 64 * CU, 16 * 64 * CU + 1])
@pytest.mark.parametrize("cell,rmax", [(3.3, 7.1), (3.05, 12.3)])
def test_forms(n, cell, rmax):
    edge = max(30.0, (n / 0.01) ** (1.0 / 3.0))
    lo = (-edge, 3.0, 0.25)
    hi = (-edge + 1.07 * edge, 3.0 + 0.93 * edge, 0.25 + edge)
    spec, xyz, types = make(n, lo, hi, cell, seed=n % 97)
    o = orc.OracleSystem(spec)
    with Simulation(spec, xyz, types, rdf=(rmax, 77)) as sim:
        sim.call_rdf_calculation()
        sim.call_rdf_calculation()
        c, frames = sim.copy_rdf_matrix()
    assert frames == 2
    assert np.array_equal(c, 2 * o.rdf_counts(xyz, types, rmax, 77, cells=True))


def test_distances_on_bin_edges():
    """Coordinates in quarter units: many distances are whole multiples of the
    bin width, where the bin is settled by the IEEE sequence."""
    spec, xyz, types = make(20_000, (0.0, 0.0, 0.0), (60.0, 60.0, 60.0), 4.0, seed=5)
    xyz = np.float32(0.25) * np.floor(xyz * 4.0).astype(np.float32)
    o = orc.OracleSystem(spec)
    for rmax, bins in ((10.0, 40), (12.5, 125), (10.0, 4000)):
        with Simulation(spec, xyz, types, rdf=(rmax, bins)) as sim:
            sim.call_rdf_calculation()
            c, _ = sim.copy_rdf_matrix()
        assert np.array_equal(c, o.rdf_counts(xyz, types, rmax, bins, cells=False)), (rmax, bins)


@pytest.mark.parametrize("scale", [1, 60])
def test_replicas_sharing_a_workgroup(scale):
    spec, boxes, counts, xyz, types = workloads.batched_replicas(12, seed=3, nmin=150, nmax=600 * scale)
    rmax = 0.4 * float(boxes[:, 1].min())
    with Simulation(spec, xyz, types, replicas=(boxes, counts), rdf=(rmax, 50)) as sim:
        sim.call_rdf_calculation()
        c, _ = sim.copy_rdf_matrix()
    off = 0
    for r, n in enumerate(counts):
        spec.box_lo, spec.box_hi = tuple(boxes[r][0::2]), tuple(boxes[r][1::2])
        ref = orc.OracleSystem(spec).rdf_counts(xyz[off:off + n], types[off:off + n], np.float32(rmax), 50,
                                                cells=False)
        assert np.array_equal(c[r], ref), r
        off += int(n)
