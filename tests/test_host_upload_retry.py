"""A call whose upload of the tables fails part of the way, and the same call
again: the second one brings up whatever the first did not.  Every allocation
and every copy of the call is made to fail in turn (CPU stand-in for the HIP
runtime; no kernel runs)."""
import pytest

from tests import hip_stub

pytestmark = hip_stub.needs_compiler

PROGRAM = """
def tables(sim):
    '''The force kernel's tables of one step: their bytes, as the GPU would read them.'''
    stub.stub_reset()
    sim.simulate(1)
    (i, *_), = launched("k_force_update")
    out = []
    for k in (6, 7, 8, 10):                 # constants, boxes, work items, external potentials
        p = stub.stub_arg(i, k)
        assert p, "table %d is null" % k
        n = stub.stub_size(p)
        assert n > 0, "table %d was freed" % k
        out.append(C.string_at(p, n))
    return out

def change(sim):
    rng = np.random.default_rng(1)
    spec, xyz, types = workloads.plain_1m(n=9000, box=200.0)
    half = np.array([[0.0, 90.0] * 3, [100.0, 200.0] * 3])
    x = np.concatenate([workloads.uniform_positions(rng, 5000, half[0, 0::2], half[0, 1::2]),
                        workloads.uniform_positions(rng, 4000, half[1, 0::2], half[1, 1::2])])
    sim.set_replicas(half, np.array([5000, 4000]), x, types[:9000])
    q = _lib.rd_pot1()
    q.type, q.subtype, q.force_const, q.radius, q.type_mask = DISK, ATTRACTIVE, 2.0, 5.0, 3
    q.normal[2] = 1.0
    assert sim.lib.rd_add_order_one_potential(sim.h, C.byref(q)) == 0

def make():
    stub.stub_reset()
    spec, xyz, types = workloads.plain_1m(n=2000, box=200.0)
    assert spec.pot1
    return Simulation(spec, xyz, types)

from readdygpu_amd import _lib
for call in (lambda s: s.initialize(), lambda s: s.simulate(0)):
    with make() as sim:
        change(sim)
        call(sim)
        want = tables(sim)
    for kind in ("malloc", "copy"):
        failures = 0
        for k in range(100):
            with make() as sim:
                change(sim)
                getattr(stub, "stub_fail_" + kind)(k)
                try:
                    call(sim)
                    break                       # no k-th one in this call
                except RdError:
                    failures += 1
                stub.stub_reset()
                call(sim)
                again = launched("k_rep_of")    # (the first attempt's launch is not counted)
                assert tables(sim) == want, (kind, k)
                assert again, "replicas of the particle indices: %s %d" % (kind, k)
        assert failures >= 3, (kind, failures)
        print(kind, failures, flush=True)
"""


def test_every_failure_is_made_good(tmp_path):
    hip_stub.run(hip_stub.build(tmp_path), PROGRAM)
