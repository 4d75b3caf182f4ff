"""When the nearest-piece grid is built: not for a few passes over pieces that
change again, once for pieces that stay, at once where the caller prepares
(rd_initialize, rd_simulate(0)) or is about to pass often (CPU stand-in for the
HIP runtime; no kernel runs)."""
import pytest

from tests import hip_stub

pytestmark = hip_stub.needs_compiler

PROGRAM = """
spec, pieces, xyz, types = workloads.learned_slab(n=1000, n_pieces=100)
rng = np.random.default_rng(1)
few = workloads.uniform_positions(rng, 50, spec.box_lo, spec.box_hi)
many = workloads.uniform_positions(rng, 600_000, spec.box_lo, spec.box_hi)
count = lambda part: len(launched(part))

def builds(before, call, times=1, pieces=pieces, combine="nearest"):
    '''Lists built by `times` calls on a handle on which `before` was called first.'''
    with Simulation(spec, xyz, types) as sim:
        def again():
            sim.set_composite(pieces, combine=combine)
        again()
        before(sim)
        stub.stub_reset()
        for _ in range(times):
            call(sim, again)
        return count("k_comp_grid")

nothing = lambda sim: None
# pieces that move before every call
assert builds(nothing, lambda s, again: (again(), s.composite_eval(few)), 20) == 0
assert builds(nothing, lambda s, again: (again(), s.gradients()), 20) == 0
assert builds(nothing, lambda s, again: (again(), s.simulate(1)), 20) == 0
# pieces that stay: once
assert builds(nothing, lambda s, again: s.composite_eval(few), 3) == 0
assert builds(nothing, lambda s, again: s.composite_eval(few), 30) == 1
assert builds(nothing, lambda s, again: s.gradients(), 30) == 1
assert builds(nothing, lambda s, again: s.simulate(1), 30) == 1
assert builds(nothing, lambda s, again: (s.simulate(1), s.gradients(), s.composite_eval(few)), 30) == 1
# many passes, or many points, in one call
assert builds(nothing, lambda s, again: (again(), s.simulate(20)), 2) == 2
assert builds(nothing, lambda s, again: (again(), s.composite_eval(many)), 2) == 2
# the caller prepares
assert builds(lambda s: s.simulate(0), lambda s, again: s.composite_eval(few)) == 0
assert builds(nothing, lambda s, again: s.simulate(0)) == 1
assert builds(nothing, lambda s, again: s.initialize()) == 1
# never
assert builds(nothing, lambda s, again: s.simulate(20), 2, combine="sum") == 0
assert builds(nothing, lambda s, again: s.simulate(20), 2, pieces=pieces[:11]) == 0
assert builds(nothing, lambda s, again: s.simulate(20), 2, pieces=pieces[:12]) == 1
assert builds(nothing, lambda s, again: s.composite_eval(many), 2, pieces=pieces[:31]) == 0
assert builds(nothing, lambda s, again: s.composite_eval(many), 2, pieces=pieces[:32]) == 1

# training data: from the boxes, and from a domain that is wider (every wave scans)
for wide, want in ((1.0, 1), (1.001, 1), (1.1, 0)):
    with Simulation(spec, xyz, types) as sim:
        sim.set_composite(pieces)
        sim.surrogate_init(1)
        sim.set_surrogate_norm(spec.box_lo, [wide * v for v in spec.box_hi], 1.0)
        stub.stub_reset()
        sim.surrogate_make_data(1_000_000)
        sim.surrogate_make_data(1_000_000)
        assert count("k_comp_grid") == want, wide
        assert count("k_sur_dataILb0ELb1E") == 2, wide          # (not the sum, the grid's kernel)

# which kernel the passes run; the captured steps follow
with Simulation(spec, xyz, types) as sim:
    sim.set_composite(pieces)
    for _ in range(3):
        sim.gradients()
    assert (count("k_composite_all"), count("k_composite_near")) == (3, 0)
    stub.stub_reset()
    sim.simulate(1)
    assert (count("k_composite_all"), count("k_composite_near")) == (0, 1)
with Simulation(spec, xyz, types) as sim:
    sim.set_composite(pieces)
    sim.simulate(2)
    stub.stub_reset()
    sim.simulate(32)
    sim.simulate(32)
    assert (count("k_composite_all"), count("k_comp_grid")) == (0, 1)
    # new boxes: built again after as many passes
    half = np.array([[0.0, spec.box_hi[0], 0.0, spec.box_hi[1], 0.0, 0.5 * spec.box_hi[2]]])
    sim.set_replicas(half, np.array([1000]), xyz * np.float32([1, 1, 0.5]), types)
    stub.stub_reset()
    sim.simulate(1)
    assert (count("k_composite_all"), count("k_comp_grid")) == (1, 0)
    sim.simulate(3)
    assert (count("k_composite_all"), count("k_composite_near"), count("k_comp_grid")) == (1, 3, 1)
"""


def test_builds(tmp_path):
    hip_stub.run(hip_stub.build(tmp_path), PROGRAM)
