"""RDF counts with large histograms against the oracle, bit for bit: both sides of
the size (32 KB) from which many particles are counted by workgroups of 1,024
threads, beyond 64 KB in every launch form, at the end of the LDS (160 KB) and
past it."""
import numpy as np
import pytest

from oracle import oracle as orc
from readdygpu_amd import Simulation, workloads
from tests.test_gpu_rdf_forms import CU, make

pytestmark = pytest.mark.gpu

# three types: 36 bytes a bin
BINS = {"32KB": 910, "32KB+": 911, "64KB+": 1821, "160KB": 4549, "global": 4550}


@pytest.mark.parametrize("bins", BINS.values(), ids=BINS)
@pytest.mark.parametrize("n", [65, 2 * 64 * CU + 1, 16 * 64 * CU + 1])
def test_forms(n, bins):
    edge = max(30.0, (n / 0.01) ** (1.0 / 3.0))
    lo = (-edge, 3.0, 0.25)
    hi = (-edge + 1.07 * edge, 3.0 + 0.93 * edge, 0.25 + edge)
    spec, xyz, types = make(n, lo, hi, 3.3, seed=n % 89)
    o = orc.OracleSystem(spec)
    with Simulation(spec, xyz, types, rdf=(6.3, bins)) as sim:
        sim.call_rdf_calculation()
        sim.call_rdf_calculation()
        c, frames = sim.copy_rdf_matrix()
    assert frames == 2
    assert np.array_equal(c, 2 * o.rdf_counts(xyz, types, 6.3, bins, cells=True))


@pytest.mark.parametrize("bins", [2000, 5000], ids=["32KB", "80KB"])
def test_replicas_sharing_a_workgroup(bins):
    """Some hundred boxes a few work items each, so that a workgroup's 512
    particles are of several."""
    spec, boxes, counts, xyz, types = workloads.batched_replicas(700, seed=3, nmin=100, nmax=2000)
    assert ((counts + 63) // 64).sum() > 16 * CU
    rmax = 0.4 * float(boxes[:, 1].min())
    with Simulation(spec, xyz, types, replicas=(boxes, counts), rdf=(rmax, bins)) as sim:
        sim.call_rdf_calculation()
        c, _ = sim.copy_rdf_matrix()
    off = 0
    for r, n in enumerate(counts):
        if r % 7 == 0:
            spec.box_lo, spec.box_hi = tuple(boxes[r][0::2]), tuple(boxes[r][1::2])
            ref = orc.OracleSystem(spec).rdf_counts(xyz[off:off + n], types[off:off + n], np.float32(rmax), bins,
                                                    cells=False)
            assert np.array_equal(c[r], ref), r
        off += int(n)
