"""Gradients and energy against the FP64 oracle on both sides of the line (3
work items of 64 particles per compute unit) up to which nine lanes share a
particle: few and many partners, every potential kind, bonds, several boxes.
Tolerances as for the smaller systems: |g - g_ref| <= 2e-5 max|g_ref| + 1e-5,
energy to 1e-5.  The oracle gets the boxes as the GPU holds them, in FP32: a bond
across the edge of a box of 174 nm differs by 3.6e-4 a bond between an edge and
its rounding (k = 50, 7.1e-6 nm)."""
import dataclasses

import numpy as np
import pytest

from oracle import oracle as orc
from readdygpu_amd import Simulation, workloads
from tests.test_gpu_parity import dense_spec, rich_spec

pytestmark = pytest.mark.gpu

LINE = 3 * 64 * 256


def oracle(spec):
    return orc.OracleSystem(dataclasses.replace(spec, box_lo=tuple(float(np.float32(v)) for v in spec.box_lo),
                                                box_hi=tuple(float(np.float32(v)) for v in spec.box_hi)))


def rich(n):
    spec = rich_spec(box=40.0 * (n / 3000.0) ** (1.0 / 3.0))[0]
    rng = np.random.default_rng(n)
    return spec, workloads.uniform_positions(rng, n, spec.box_lo, spec.box_hi), rng.integers(0, 3, n).astype(np.int32)


MODELS = {"dense": lambda n: dense_spec(n=n, box=22.0 * (n / 6000.0) ** (1.0 / 3.0)),        # 36 partners
          "denser": lambda n: dense_spec(n=n, box=22.0 * (n / 14000.0) ** (1.0 / 3.0)),      # 84
          "rich": rich,
          "chains": lambda n: workloads.bonded_chains(n // 8, 8, box=120.0 * (n / 16000.0) ** (1.0 / 3.0)),
          "confined": lambda n: workloads.plain_1m(n=n, box=1000.0 * (n / 1e6) ** (1.0 / 3.0))}


@pytest.mark.parametrize("n", [LINE, LINE + 8])
@pytest.mark.parametrize("make", MODELS.values(), ids=MODELS)
def test_against_fp64(make, n):
    spec, xyz, types = make(n)
    o = oracle(spec)
    with Simulation(spec, xyz, types) as sim:
        g, e = sim.gradients()
    gr, er = o.gradients(xyz.astype(np.float64), types)
    assert np.abs(g - gr).max() <= 2e-5 * np.abs(gr).max() + 1e-5, np.abs(g - gr).max()
    assert abs(e - er) <= 1e-5 * max(1.0, abs(er))


def test_boxes_past_the_line():
    spec, boxes, counts, xyz, types = workloads.batched_replicas(40, seed=8, nmin=500, nmax=6000)
    assert ((counts + 63) // 64).sum() > 3 * 256
    with Simulation(spec, xyz, types, replicas=(boxes, counts)) as sim:
        g, e = sim.gradients()
    total, off = 0.0, 0
    for b, n in zip(boxes, counts):
        spec.box_lo, spec.box_hi = tuple(b[0::2]), tuple(b[1::2])
        gr, er = oracle(spec).gradients(xyz[off:off + n].astype(np.float64), types[off:off + n])
        assert np.abs(g[off:off + n] - gr).max() <= 2e-5 * np.abs(gr).max() + 1e-5
        total, off = total + er, off + n
    assert abs(e - total) <= 1e-5 * max(1.0, abs(total))
