"""Pair sets where a particle has more partners than are kept between the two
kernels (four), at sizes on both sides of the launch rule, bit for bit against
the oracle; and the allocation-free candidates, which keep none."""
import numpy as np
import pytest

from oracle import oracle as orc
from readdygpu_amd import Simulation, workloads
from tests.test_gpu_parity import dense_spec, rich_spec

pytestmark = pytest.mark.gpu

CU = 256


@pytest.mark.parametrize("make", [lambda: dense_spec(n=3000), lambda: dense_spec(n=14000), rich_spec,
                                  lambda: rich_spec(cell=2.3), lambda: rich_spec(cell=14.0),
                                  lambda: workloads.plain_1m(n=16 * 64 * CU, box=640.0),
                                  lambda: workloads.plain_1m(n=16 * 64 * CU + 65, box=640.0)],
                         ids=["dense", "denser", "rich", "three_cell_stencil", "tiny_lattice", "at_rule", "past_rule"])
def test_pairs_and_candidates(make):
    spec, xyz, types = make()
    nt = spec.n_types
    if spec.reaction_radii is None:
        spec.reaction_radii = np.full((nt, nt), 1.5)
    o = orc.OracleSystem(spec)
    with Simulation(spec, xyz, types) as sim:
        for _ in range(2):                       # the buffers are used again
            assert np.array_equal(sim.neighbor_pairs(), o.pairs(xyz, types))
            c = o.candidates(xyz, types)
            assert np.array_equal(sim.reaction_candidates(), c)
            assert np.array_equal(sim.reaction_candidates_noalloc(len(c) + 5), c)


def test_sizes_up_to_one_item():
    for n in (1, 2, 5, 63, 64, 65):
        spec, xyz, types = dense_spec(n=n, box=6.0 if n < 10 else 9.0)
        o = orc.OracleSystem(spec)
        with Simulation(spec, xyz, types) as sim:
            assert np.array_equal(sim.neighbor_pairs(), o.pairs(xyz, types, brute=True)), n
