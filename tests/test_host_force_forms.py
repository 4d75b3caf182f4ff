"""Which kernel a step and a gradient run, for the systems by which the forms of
the force kernel are tested and on both sides of each rule (CPU stand-in for the
HIP runtime with 256 compute units; no kernel runs)."""
import pytest

from tests import hip_stub

pytestmark = hip_stub.needs_compiler

PROGRAM = """
import pytest
from tests import test_gpu_dealt_hits as dealt, test_gpu_sparse_lists as sparse, test_gpu_overflow_forms as overflow

CU = 256
SPARSE, DEALT, ROWS, LANES9, LANES3 = ("k_force_update_sparse", "k_force_update_dealt", "k_force_updateILi256",
                                       "k_force_update_spreadILi9E", "k_force_update_spreadILi3E")

def step(spec, xyz, types, replicas=None, **launch):
    with Simulation(spec, xyz, types, replicas=replicas) as sim:
        if launch:
            sim.set_launch_config(**launch)
        stub.stub_reset()
        sim.simulate(1)
        (i, name, *_), = launched("k_force_update")
        return name

def is_form(name, form):
    return form + ("" if "ILi" in form else "PK") in name        # (mangled: the form, then the arguments)

def cases(module):
    '''Box cases of the module's tests'''
    (mark,) = [m for m in module.test_boxes.pytestmark if m.name == "parametrize"]
    return mark.args[1]

def boxes_form(cells, nmin, nmax, clump):
    spec, bounds, counts, xyz, types = dealt.boxes(cells, nmin, nmax, clump)
    return step(spec, xyz, types, (bounds, counts))

# the box cases of both tests: by the mean number of candidates (27 n / cells)
# and of partners, and by the number of cells per axis
want = {((3, 3, 3), 1, 1, 1.0): SPARSE, ((2, 3, 3), 20, 70, 1.0): ROWS, ((8, 8, 8), 80, 80, 1.0): SPARSE,
        ((8, 8, 8), 96, 96, 1.0): DEALT, ((12, 12, 12), 200, 300, 0.25): SPARSE, ((2, 9, 9), 20, 30, 1.0): ROWS}
for module, default in ((dealt, DEALT), (sparse, SPARSE)):
    for case in cases(module):
        form = want.get(tuple(case), default)
        name = boxes_form(*case)
        assert is_form(name, form), (module.__name__, case, name)

# single-particle waves of the dealt form
for nmin, nmax in ((65, 65), (129, 129)):
    assert is_form(boxes_form((3, 3, 3), nmin, nmax, 1.0), DEALT)

# lanes per particle: 3 and 8 work items per compute unit
for n, form in ((1, LANES9), (3 * 64 * CU, LANES9), (3 * 64 * CU + 1, LANES3), (8 * 64 * CU, LANES3)):
    assert is_form(step(*workloads.plain_1m(n=n, box=max(30.0, 1000.0 * (n / 1e6) ** (1 / 3)))), form), n
n = 8 * 64 * CU + 1
assert is_form(step(*workloads.plain_1m(n=n, box=1000.0 * (n / 1e6) ** (1 / 3))), ROWS)
assert "spread" not in step(*workloads.plain_1m(n=1000, box=100.0), block=128)

# the systems of the overflow test
for form, name in (("lanes9", LANES9), ("lanes3", LANES3), ("sparse", SPARSE), ("rows", ROWS), ("dealt", DEALT),
                   ("dealt_idle_lane", DEALT)):
    got = step(*overflow.system(form, True))
    assert is_form(got, name), (form, got)

# gradients
for n, part in ((3 * 64 * CU, "k_gradients_spread"), (3 * 64 * CU + 1, "k_gradientsPK")):
    spec, xyz, types = workloads.plain_1m(n=n, box=400.0)
    with Simulation(spec, xyz, types) as sim:
        stub.stub_reset()
        sim.gradients()
        (i, name, *_), = launched("k_gradients")
        assert part in name, (n, name)
"""


def test_forms(tmp_path):
    hip_stub.run(hip_stub.build(tmp_path), PROGRAM)
