"""Runs of steps in chunks of 256 and 16, launched or as graphs: the same
trajectory as step by step, in a first call, a repeated one and after new
particles."""
import numpy as np
import pytest

from readdygpu_amd import Simulation, workloads

pytestmark = pytest.mark.gpu


def test_lengths():
    spec, xyz, types = workloads.plain_10k(n=300)
    lengths = [15, 16, 17, 95, 96, 97, 255, 256, 257, 600, 2047, 2048, 2145]
    ref = {0: xyz}
    with Simulation(spec, xyz, types) as sim:
        for k in range(1, 2 * max(lengths) + 1):
            sim.simulate(1)
            if k in lengths or k % 2 == 0 and k // 2 in lengths:
                ref[k] = sim.copy_pos_from_device()[0].copy()
    with Simulation(spec, xyz, types) as sim:
        for n in lengths:
            sim.set_particles(xyz, types)
            sim.set_step(0)
            for times in (1, 2):
                sim.simulate(n)
                assert np.array_equal(sim.copy_pos_from_device()[0], ref[times * n]), (n, times)
            assert sim.info().step == 2 * n and sim.check_invariants() == 0
