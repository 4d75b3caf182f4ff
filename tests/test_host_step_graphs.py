"""When steps are captured as graphs: never for a few steps on tables that
change again, once for lengths that repeat, and inside a first call only if it
is long (CPU stand-in for the HIP runtime; no kernel runs)."""
import pytest

from tests import hip_stub

pytestmark = hip_stub.needs_compiler

PROGRAM = """
spec, xyz, types = workloads.plain_10k(n=2000)

def frames(steps, change, times=5):
    '''Per call: captures, graph launches, force-kernel launches (captured ones among them).'''
    out = []
    with Simulation(spec, xyz, types) as sim:
        for _ in range(times):
            if change:
                sim.set_particles(xyz, types)
            stub.stub_reset()
            sim.simulate(steps)
            out.append((stub.stub_captures(), stub.stub_graph_launches(), len(launched("k_force_update"))))
    return out

# particles that change before every call: launched, except where the call itself is long
for steps in (1, 15, 16, 17, 32, 48, 80, 95):
    assert set(frames(steps, True)) == {(0, 0, steps)}, steps
assert set(frames(96, True)) == {(1, 5, 16 + 16)}                   # a chunk, then the graph five times
assert set(frames(100, True)) == {(1, 5, 16 + 16 + 4)}
assert set(frames(512, True)) == {(1, 31, 32)}                      # (no graph of 256)
assert set(frames(2047, True)) == {(1, 126, 32 + 15)}
assert set(frames(2048, True)) == {(1, 7, 512)}                     # one of 256
assert set(frames(2048 + 97, True)) == {(2, 7 + 5, 512 + 32 + 1)}

# the same particles: the second call captures, later ones launch graphs
assert frames(15, False) == [(0, 0, 15)] * 5
assert frames(16, False) == [(0, 0, 16), (1, 1, 16)] + [(0, 1, 0)] * 3
assert frames(20, False) == [(0, 0, 20), (1, 1, 16 + 4)] + [(0, 1, 4)] * 3
assert frames(300, False) == [(1, 17, 32 + 12), (1, 1 + 2, 256 + 12)] + [(0, 3, 12)] * 3
"""


def test_captures(tmp_path):
    hip_stub.run(hip_stub.build(tmp_path), PROGRAM)
