"""Workloads that a user of this framework has it do, each through the public
entry points of ``readdygpu_amd.Simulation``, for timing and comparison.

The cases are the frames of Brownian-dynamics runs (steps, then what the
program reads back), the analysis of a frame, reactions between frames, forces,
and the learned external potential (training and evaluation), over the sizes
of ``readdygpu_amd.workloads``.  A handle's state moves on from pass to pass,
as it does in a run.

Kinds (``case["kind"]``):
  plain      two species with harmonic repulsion in a periodic box
  confined   four species, repulsion + a piecewise well, spherical confinement
  replicas   independent boxes of different size in one handle
  cytosol    crowded eight-species boxes with a membrane of disks
  slab       a slab with a composite potential, exact or through the surrogate
  chains     bonded chains
  reactive   steps, candidates, positions and reactions between frames
  sets       RDF, neighbour pairs and reaction candidates of a frame
  gradients  forces and energy of a frame
  learn      training data, surrogate training and validation
  points     composite and surrogate at given points
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from readdygpu_amd import Simulation, workloads
from readdygpu_amd.model import CYLINDER

MLP_SHAPES = [(64, 3), (64,), (64, 64), (64,), (64, 64), (64,), (3, 64), (3,)]


def listed():
    return [
        # the smallest call: one step of a small box, positions read after it
        # (a program that steers or watches every step)
        {"name": "call_2k", "kind": "plain", "n": 2000, "steps": 1, "rdf_bins": 0},
        # the 10,000-particle workload's own frame: 100 steps, RDF 0-20 nm in 200 bins
        {"name": "frame_10k", "kind": "plain", "n": 10_000, "steps": 100, "rdf_bins": 200},
        # the 1M-particle workload: 100 steps, then the frame hand-off
        {"name": "frame_1m", "kind": "confined", "n": 1_000_000, "steps": 100},
        # batched replicas of 500-50,000 particles
        {"name": "replicas_64", "kind": "replicas", "replicas": 64, "nmin": 500, "nmax": 50_000, "steps": 50},
        # crowded cytosol boxes, exact membrane of 256 disks on two of eight species
        {"name": "cytosol_16", "kind": "cytosol", "replicas": 16, "nmin": 20_000, "nmax": 200_000, "pieces": 256,
         "steps": 20},
        # slab with the exact composite of 512 pieces (all species feel it)
        {"name": "slab_exact", "kind": "slab", "n": 500_000, "pieces": 512, "combine": "nearest", "surrogate": False,
         "steps": 20},
        # the 2M slab with the surrogate in the composite's place
        {"name": "slab_surrogate", "kind": "slab", "n": 2_000_000, "pieces": 512, "combine": "nearest",
         "surrogate": True, "steps": 20},
        # bonded chains: 2,000 chains of 8 beads, 100 steps per frame
        {"name": "chains_16k", "kind": "chains", "chains": 2000, "length": 8, "steps": 100},
        # the reaction loop: 20 steps, candidates, positions, up to 100 pairs of
        # A+B react (they swap species, so that the composition stays)
        {"name": "reactive_100k", "kind": "reactive", "n": 100_000, "steps": 20, "events": 100},
        # the analysis of a 1M-particle frame
        {"name": "sets_1m", "kind": "sets", "n": 1_000_000, "rdf_bins": 200},
        # forces and energy of a frame
        {"name": "gradients_200k", "kind": "gradients", "n": 200_000},
        # learning a composite: training data, 256 optimiser steps of 8,192
        # samples, validation
        {"name": "learn_512", "kind": "learn", "pieces": 512, "combine": "nearest", "samples": 1_000_000,
         "batch": 8192, "steps": 256, "validate": 200_000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["plain", "confined", "replicas", "cytosol", "slab", "chains", "reactive", "sets", "gradients",
                       "learn", "points"])
    if kind == "plain":
        return {"kind": kind, "n": _log_int(rng, 1000, 100_000), "steps": _log_int(rng, 1, 100),
                "rdf_bins": rng.choice([0, 100, 200])}
    if kind == "confined":
        return {"kind": kind, "n": _log_int(rng, 20_000, 1_000_000), "steps": _log_int(rng, 5, 100)}
    if kind == "replicas":
        return {"kind": kind, "replicas": _log_int(rng, 2, 64), "nmin": 500, "nmax": _log_int(rng, 2000, 50_000),
                "steps": _log_int(rng, 5, 50)}
    if kind == "cytosol":
        return {"kind": kind, "replicas": _log_int(rng, 2, 16), "nmin": 20_000, "nmax": _log_int(rng, 30_000, 200_000),
                "pieces": _log_int(rng, 16, 256), "steps": _log_int(rng, 2, 20)}
    if kind == "slab":
        surrogate = rng.random() < 0.5
        combine = "nearest" if surrogate or rng.random() < 0.5 else "sum"
        # (the sum of many pieces is too stiff for the slab's time step)
        pieces = _log_int(rng, 2, 512) if combine == "nearest" else rng.randint(2, 8)
        return {"kind": kind, "n": _log_int(rng, 30_000, 2_000_000 if surrogate else 500_000), "pieces": pieces,
                "combine": combine, "surrogate": surrogate, "steps": _log_int(rng, 2, 20)}
    if kind == "chains":
        return {"kind": kind, "chains": _log_int(rng, 50, 2000), "length": rng.randint(2, 8),
                "steps": _log_int(rng, 5, 100)}
    if kind == "reactive":
        return {"kind": kind, "n": _log_int(rng, 10_000, 100_000), "steps": _log_int(rng, 2, 20),
                "events": _log_int(rng, 1, 100)}
    if kind == "sets":
        return {"kind": kind, "n": _log_int(rng, 20_000, 1_000_000), "rdf_bins": rng.choice([50, 100, 200])}
    if kind == "gradients":
        return {"kind": kind, "n": _log_int(rng, 5000, 200_000)}
    combine = rng.choice(["nearest", "sum"])
    if kind == "learn":
        return {"kind": kind, "pieces": _log_int(rng, 1, 512), "combine": combine,
                "samples": _log_int(rng, 20_000, 1_000_000), "batch": _log_int(rng, 256, 8192),
                "steps": _log_int(rng, 20, 256), "validate": _log_int(rng, 10_000, 200_000)}
    return {"kind": kind, "pieces": _log_int(rng, 1, 512), "combine": combine, "points": _log_int(rng, 1000, 300_000)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _weights(seed):
    """Untrained network: uniform(-a, a), a = sqrt(6 / fan_in), biases 0."""
    rng = np.random.default_rng(seed)
    parts = []
    for s in MLP_SHAPES:
        parts.append(rng.uniform(-1.0, 1.0, s) * math.sqrt(6.0 / s[1]) if len(s) == 2 else np.zeros(s))
    return np.concatenate([p.reshape(-1) for p in parts]).astype(np.float32)


def _in_boxes(boxes, counts, seed):
    """Positions of the seed in the (case's own) replica boxes."""
    rng = np.random.default_rng(seed)
    return np.concatenate([workloads.uniform_positions(rng, int(n), b[0::2], b[1::2]) for b, n in zip(boxes, counts)])


def _model(case, seed):
    """The model and coordinates of a case: a dict with spec, xyz, types and,
    where it has them, replica boxes, pieces and the types they act on."""
    kind = case["kind"]
    if kind == "plain":
        spec, xyz, types = workloads.plain_10k(n=case["n"], seed=seed)
        return {"spec": spec, "xyz": xyz, "types": types}
    if kind in ("confined", "reactive", "sets", "gradients"):
        n = case["n"]
        spec, xyz, types = workloads.plain_1m(n=n, seed=seed, box=1000.0 * (n / 1e6) ** (1.0 / 3.0))
        return {"spec": spec, "xyz": xyz, "types": types}
    if kind == "replicas":
        spec, boxes, counts, _, types = workloads.batched_replicas(case["replicas"], nmin=case["nmin"],
                                                                   nmax=case["nmax"])
        spec.seed = seed
        return {"spec": spec, "xyz": _in_boxes(boxes, counts, seed), "types": types, "replicas": (boxes, counts)}
    if kind == "cytosol":
        spec, boxes, counts, _, types, pieces, mtypes = workloads.crowded_cytosol(
            case["replicas"], nmin=case["nmin"], nmax=case["nmax"], n_pieces=case["pieces"])
        spec.seed = seed
        return {"spec": spec, "xyz": _in_boxes(boxes, counts, seed), "types": types, "replicas": (boxes, counts),
                "pieces": pieces, "mtypes": mtypes}
    if kind == "chains":
        box = 120.0 * (case["chains"] * case["length"] / 16_000.0) ** (1.0 / 3.0)
        spec, xyz, types = workloads.bonded_chains(case["chains"], case["length"], box=max(box, 20.0), seed=seed)
        return {"spec": spec, "xyz": xyz, "types": types}
    # slab, learn, points: the slab's density (2M particles in 2000 x 2000 nm)
    n = case.get("n", 1000)
    edge = 2000.0 * math.sqrt(n / 2e6) if kind == "slab" else 2000.0
    spec, pieces, xyz, types = workloads.learned_slab(n=n, seed=seed, n_pieces=case["pieces"],
                                                      box=(edge, edge, 400.0))
    if case["combine"] == "sum" and kind == "slab":
        for p in pieces:      # a summed disk pulls at any distance: weak pieces keep the step stable
            p.k = 0.05
    return {"spec": spec, "xyz": xyz, "types": types, "pieces": pieces}


def prepare(case, seed):
    kind = case["kind"]
    m = _model(case, seed)
    spec = m["spec"]
    rdf = (20.0, case["rdf_bins"]) if case.get("rdf_bins") else None
    if rdf and kind == "sets":      # (a small frame's box may be narrower than the range)
        rdf = (min(20.0, 0.49 * spec.box_hi[0]), rdf[1])
    sim = Simulation(spec, m["xyz"], m["types"], rdf=rdf, replicas=m.get("replicas"))
    state = {"case": case, "sim": sim}
    if "pieces" in m:
        sim.set_composite(m["pieces"], types=m.get("mtypes"), combine=case.get("combine", "nearest"))
        if case.get("surrogate") or kind in ("learn", "points"):
            state["weights"] = _weights(seed)
            sim.set_surrogate_weights(state["weights"])
            sim.set_surrogate_norm(spec.box_lo, spec.box_hi, 1.0)
        if case.get("surrogate"):
            sim.set_external_mode(True)
        sim.simulate(0)             # the tables go to the GPU
    if kind == "learn":
        state["seed"] = seed
    if kind == "sets":
        # the caller's own pair buffers, unused entries -1
        state["pairs"] = np.full((case["n"] // 2 + 1000, 2), -1, np.int64)
        state["candidates"] = np.full((case["n"] // 20 + 1000, 2), -1, np.int64)
    if kind == "points":
        rng = np.random.default_rng(seed + 1)
        state["xyz"] = workloads.uniform_positions(rng, case["points"], spec.box_lo, spec.box_hi)
        span = np.asarray(spec.box_hi, np.float32)
        state["xn"] = (state["xyz"] * (2.0 / span) - 1.0).astype(np.float32)
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    case, sim = state["case"], state["sim"]
    kind = case["kind"]
    if kind in ("plain", "chains"):
        # frame loop with the synchronous copy
        sim.simulate(case["steps"])
        out = {}
        if case.get("rdf_bins"):
            sim.call_rdf_calculation()
            out["counts"] = sim.copy_rdf_matrix()[0].view(np.int64)
        out["xyz"] = sim.copy_pos_from_device()[0]
        return out
    if kind in ("confined", "replicas", "cytosol", "slab"):
        # frame loop with the pinned hand-off
        sim.simulate_async(case["steps"])
        sim.frame_copy()
        xyz, types = sim.frame_wait()
        return {"xyz": xyz, "types": types}
    if kind == "reactive":
        sim.simulate(case["steps"])
        pairs = sim.reaction_candidates()
        xyz, types = sim.copy_pos_from_device()
        # pairs whose particles take part in no earlier pair
        flat = pairs.reshape(-1)
        first = np.zeros(len(flat), bool)
        first[np.unique(flat, return_index=True)[1]] = True
        chosen = pairs[first.reshape(-1, 2).all(1)][:case["events"]].reshape(-1)
        entries = np.zeros((len(chosen), 6), np.float32)
        entries[:, 0] = chosen
        entries[:, 1] = 1 - types[chosen]       # species 0 and 1 change places
        entries[:, 2:5] = xyz[chosen]
        entries[:, 5] = chosen
        sim.apply_reactions(np.concatenate([np.array([len(chosen)], np.float32), entries.reshape(-1)]))
        xyz, types = sim.copy_pos_from_device()
        reported = np.full((case["n"] // 10 + 64, 2), -1, np.int64)
        reported[:len(pairs)] = pairs[:len(reported)]
        return {"pairs": reported, "xyz": xyz, "types": types}
    if kind == "sets":
        sim.call_rdf_calculation()
        counts, frames = sim.copy_rdf_matrix()
        out = {"counts": counts.view(np.int64), "frames": frames}
        for name, entry in (("pairs", sim.lib.rd_neighbor_pairs), ("candidates", sim.lib.rd_reaction_candidates)):
            found = ctypes.c_long()
            buf = out[name] = state[name]
            if entry(sim.h, buf.ctypes.data_as(ctypes.c_void_p), len(buf), ctypes.byref(found)) != 0:
                raise RuntimeError(name)
            out["n_" + name] = found.value
        return out
    if kind == "gradients":
        g, e = sim.gradients()
        return {"grad": g, "energy": np.array([e])}
    if kind == "learn":
        # sample the composite, train from the given weights, validate
        gscale = sim.surrogate_make_data(case["samples"], seed=state["seed"] + 1)
        sim.set_surrogate_weights(state["weights"])
        curve = sim.surrogate_train(case["steps"], batch=case["batch"], seed=state["seed"] + 2)
        rmse = sim.surrogate_validate(case["validate"], seed=state["seed"] + 3)
        return {"gscale": gscale, "curve": curve, "weights": sim.surrogate_weights(), "rmse": rmse}
    g, e = sim.composite_eval(state["xyz"])
    return {"grad": g, "energy": e, "y": sim.surrogate_predict(state["xn"])}


# ---------------------------------------------------------------------------
# the work that a pass cannot do without
# ---------------------------------------------------------------------------
def _particles(case):
    if "n" in case:
        return case["n"]
    if "chains" in case:
        return case["chains"] * case["length"]
    # replica sizes are log-uniform
    return case["replicas"] * (case["nmax"] - case["nmin"]) / math.log(case["nmax"] / case["nmin"])


MLP_FLOPS = 2 * 8576
STEP_FLOPS = 200      # noise, displacement and wrap of a particle, and its few interacting partners


def work(case):
    kind = case["kind"]
    if kind == "points":
        m = case["points"]
        evals = case["pieces"] if case["combine"] == "sum" else 1
        return {"bytes": m * (12 + 16 + 12 + 12), "flops": m * (25 * evals + MLP_FLOPS)}
    if kind == "learn":
        evals = case["pieces"] if case["combine"] == "sum" else 1
        sampled = case["samples"] + case["validate"]
        trained = case["steps"] * case["batch"]
        return {"bytes": 24 * sampled + 24 * trained,
                "flops": 25 * evals * sampled + MLP_FLOPS * (3 * trained + case["validate"])}
    n = _particles(case)
    if kind == "gradients":
        return {"bytes": 28 * n, "flops": 100 * n}
    if kind == "sets":
        # 16 B in; partners within 20 nm (33.5 at 1e-3 per nm^3, each met once)
        # for the RDF, 0.24 neighbour pairs out
        return {"bytes": 16 * n + 16 * 0.24 * n + 16 * 16 * case["rdf_bins"], "flops": n * 17 * 10}
    per_step = {"bytes": 28 * n, "flops": STEP_FLOPS * n}
    if kind in ("cytosol", "slab"):
        acts = 0.25 if kind == "cytosol" else 1.0
        evals = case["pieces"] if case.get("combine") == "sum" else 1
        per_step["flops"] += acts * n * (MLP_FLOPS if case.get("surrogate") else 25 * evals)
    out = 16 * n
    return {"bytes": case["steps"] * per_step["bytes"] + out, "flops": case["steps"] * per_step["flops"]}


# ---------------------------------------------------------------------------
# the same in 64 bits, without this repository's code
# ---------------------------------------------------------------------------
_M32 = 0xFFFFFFFF


def _mul32(a, m):
    """High and low words of the 64-bit products of 32-bit values."""
    lo = (a * (m & 0xFFFF)) + (((a * (m >> 16)) & 0xFFFF) << 16)
    hi = (a * (m >> 16) + ((a * (m & 0xFFFF)) >> 16)) >> 16
    return hi, lo & _M32


def _normals(seed, stream, step, index):
    """Three N(0,1) values per particle: Philox4x32-10 of (index, step, stream), then Box-Muller."""
    c = [index, torch.full_like(index, step & _M32), torch.full_like(index, (step >> 32) ^ ((stream << 16) & _M32)),
         torch.full_like(index, 0x52444E53)]
    k0, k1 = seed & _M32, (seed >> 32) & _M32
    for r in range(10):
        if r:
            k0, k1 = (k0 + 0x9E3779B9) & _M32, (k1 + 0xBB67AE85) & _M32
        h0, l0 = _mul32(c[0], 0xD2511F53)
        h1, l1 = _mul32(c[2], 0xCD9E8D57)
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
    s = 2.0 ** -24
    a1, a2 = ((c[0] >> 8) + 1).double() * s, (c[1] >> 8).double() * s
    b1, b2 = ((c[2] >> 8) + 1).double() * s, (c[3] >> 8).double() * s
    ra, rb = torch.sqrt(-2.0 * torch.log(a1)), torch.sqrt(-2.0 * torch.log(b1))
    t = 2.0 * math.pi
    return torch.stack([ra * torch.cos(t * a2), ra * torch.sin(t * a2), rb * torch.cos(t * b2)], 1)


def _pairs(x, lo, box, reach):
    """Index pairs (i, j), i != j both ways, that may lie within `reach` (minimum image), in parts."""
    n = len(x)
    cells = [int(b // (reach * 1.0001)) for b in box]
    if min(cells) < 3 or n < 400:
        step = max(1, 4_000_000 // n)
        every = torch.arange(n, device=x.device)
        for i0 in range(0, n, step):
            i, j = torch.meshgrid(every[i0:i0 + step], every, indexing="ij")
            off = i != j
            yield i[off], j[off]
        return
    size = torch.tensor(cells, device=x.device)
    at = ((x - lo) / box * size).long().clamp_(min=0)
    at = torch.minimum(at, size - 1)
    key = (at[:, 2] * cells[1] + at[:, 1]) * cells[0] + at[:, 0]
    order = torch.argsort(key)
    count = torch.bincount(key, minlength=cells[0] * cells[1] * cells[2])
    start = torch.cumsum(count, 0) - count
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                b = (at + torch.tensor([dx, dy, dz], device=x.device)) % size
                k = (b[:, 2] * cells[1] + b[:, 1]) * cells[0] + b[:, 0]
                c, s = count[k], start[k]
                i = torch.nonzero(c > 0)[:, 0]
                q = 0
                while len(i):
                    j = order[s[i] + q]
                    off = i != j
                    yield i[off], j[off]
                    q += 1
                    i = i[c[i] > q]


def _pair_terms(spec, device):
    """Per potential: its parameters and the type pairs it acts on."""
    r0 = torch.tensor(spec.radius_sum(), dtype=torch.float64, device=device)
    pots = [(p, torch.tensor(spec.pot2_mask(p).astype(bool), device=device)) for p in spec.pot2]
    return r0, pots


def _forces(spec, x, t, lo, box, energy=False):
    """Gradient of the pair, bond and confinement terms, and their energy."""
    g = torch.zeros_like(x)
    e = torch.zeros((), dtype=torch.float64, device=x.device)
    r0_of, pots = _pair_terms(spec, x.device)
    reach = float(spec.pair_range().max())
    for i, j in _pairs(x, lo, box, reach):
        d = x[i] - x[j]
        d = d - box * torch.round(d / box)
        d2 = (d * d).sum(1)
        near = (d2 < reach * reach) & (d2 > 0)
        i, j, d, r = i[near], j[near], d[near], torch.sqrt(d2[near])
        ti, tj = t[i], t[j]
        r0 = r0_of[ti, tj]
        pre = torch.zeros_like(r)
        for p, acts in pots:
            if p.kind == 1:         # harmonic repulsion
                on = acts[ti, tj] & (r < r0) & (r <= spec.max_cutoff)
                pre += torch.where(on, p.k * (r - r0) / r, 0.0)
                u = torch.where(on, 0.5 * p.k * (r - r0) ** 2, 0.0)
            else:                   # piecewise harmonic well
                l, wc = p.length, p.depth / (0.25 * p.length ** 2)
                on = acts[ti, tj] & (r < r0 + l) & (r <= spec.max_cutoff)
                a, b = r < r0, r < r0 + 0.5 * l
                v = torch.where(a, p.k * (r - r0), torch.where(b, wc * (r - r0), -wc * (r - r0 - l)))
                pre += torch.where(on, v / r, 0.0)
                u = torch.where(a, 0.5 * p.k * (r - r0) ** 2 - p.depth,
                                torch.where(b, 0.5 * wc * (r - r0) ** 2 - p.depth, -0.5 * wc * (r - r0 - l) ** 2))
                u = torch.where(on, u, 0.0)
            if energy:
                e = e + 0.5 * u.sum()
        g.index_add_(0, i, pre[:, None] * d)
    if spec.bonds is not None:
        i, j = torch.tensor(spec.bonds, dtype=torch.long, device=x.device).T
        d = x[i] - x[j]
        d = d - box * torch.round(d / box)
        r = torch.sqrt((d * d).sum(1))
        f = (spec.bond_pots[0].k * (1.0 - r0_of[t[i], t[j]] / r))[:, None] * d
        g.index_add_(0, i, f)
        g.index_add_(0, j, -f)
    for p in spec.pot1:             # attractive sphere
        v = x - torch.tensor(p.origin, dtype=torch.float32, device=x.device).double()
        d = torch.sqrt((v * v).sum(1))
        out = torch.clamp(d - float(np.float32(p.radius)), min=0.0)
        g += (p.k * out / d)[:, None] * v
        e = e + 0.5 * p.k * (out * out).sum()
    return g, e


def _composite(pieces, combine, x):
    """Gradient and energy of z-normal attractive disks and cylinders."""
    dev = x.device
    o = torch.tensor([p.origin for p in pieces], dtype=torch.float32, device=dev).double()
    R = torch.tensor([p.radius for p in pieces], dtype=torch.float32, device=dev).double()
    hh = torch.tensor([0.5 * p.height if p.kind == CYLINDER else 0.0 for p in pieces], dtype=torch.float32,
                      device=dev).double()
    k = torch.tensor([p.k for p in pieces], dtype=torch.float32, device=dev).double()
    grads, energies = [], []
    for part in torch.split(x, max(1, 8_000_000 // len(pieces))):
        v = part[:, None, :] - o[None]
        r = torch.sqrt(v[..., 0] ** 2 + v[..., 1] ** 2)
        dn, dr = torch.clamp(v[..., 2].abs() - hh, min=0.0), torch.clamp(r - R, min=0.0)
        u = 0.5 * k * (dn * dn + dr * dr)
        s = torch.where(r > 0, k * dr / torch.clamp(r, min=1e-300), torch.zeros_like(r))
        f = torch.stack([s * v[..., 0], s * v[..., 1], k * dn * torch.sign(v[..., 2])], -1)
        if combine == "sum":
            grads.append(f.sum(1))
            energies.append(u.sum(1))
        else:
            b = torch.argmin(u, 1, keepdim=True)
            grads.append(torch.gather(f, 1, b[..., None].expand(-1, 1, 3))[:, 0])
            energies.append(torch.gather(u, 1, b)[:, 0])
    return torch.cat(grads), torch.cat(energies)


def _network(w, xn):
    parts, at = [], 0
    for s in MLP_SHAPES:
        size = int(np.prod(s))
        parts.append(torch.tensor(w[at:at + size].reshape(s), dtype=torch.float64, device=xn.device))
        at += size
    h = xn
    for layer in range(4):
        h = h @ parts[2 * layer].T + parts[2 * layer + 1]
        if layer < 3:
            h = h * torch.sigmoid(h)
    return h


def exact(case, seed):
    kind = case["kind"]
    if kind in ("reactive", "sets", "learn"):
        return None                 # whole numbers, or a training run
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    m = _model(case, seed)
    spec = m["spec"]
    if kind == "points":
        rng = np.random.default_rng(seed + 1)
        xyz = workloads.uniform_positions(rng, case["points"], spec.box_lo, spec.box_hi)
        g, e = _composite(m["pieces"], case["combine"], torch.tensor(xyz, device=dev).double())
        xn = (xyz * (2.0 / np.asarray(spec.box_hi, np.float32)) - 1.0).astype(np.float32)
        y = _network(_weights(seed), torch.tensor(xn, device=dev).double())
        return {"grad": g, "energy": e, "y": y}
    if "replicas" in m:
        boxes, counts = m["replicas"]
    else:
        boxes = np.array([[v for d in range(3) for v in (spec.box_lo[d], spec.box_hi[d])]])
        counts = [len(m["xyz"])]
    D = torch.tensor([t.D for t in spec.types], dtype=torch.float64, device=dev)
    acts = torch.tensor([t in m.get("mtypes", range(spec.n_types)) for t in range(spec.n_types)], device=dev)
    done, parts = 0, []
    for r, n in enumerate(counts):
        n = int(n)
        stream = r if "replicas" in m else spec.stream
        x = torch.tensor(m["xyz"][done:done + n], device=dev).double()
        t = torch.tensor(m["types"][done:done + n], dtype=torch.long, device=dev)
        done += n
        lo = torch.tensor(boxes[r][0::2].copy(), dtype=torch.float32, device=dev).double()
        box = torch.tensor(boxes[r][1::2].copy(), dtype=torch.float32, device=dev).double() - lo
        if kind == "gradients":
            g, e = _forces(spec, x, t, lo, box, energy=True)
            return {"grad": g, "energy": e.reshape(1)}
        index = torch.arange(n, device=dev)
        a, b = (spec.dt * D / spec.kbt)[t][:, None], torch.sqrt(2.0 * D * spec.dt)[t][:, None]
        for step in range(case["steps"]):
            g, _ = _forces(spec, x, t, lo, box)
            if case.get("surrogate"):
                g = g + torch.where(acts[t][:, None], _network(_weights(seed), 2.0 * (x - lo) / box - 1.0), 0.0)
            elif "pieces" in m:
                on = torch.nonzero(acts[t])[:, 0]
                g.index_add_(0, on, _composite(m["pieces"], case.get("combine", "nearest"), x[on])[0])
            x = x - a * g + b * _normals(spec.seed, stream, step, index)
            x = torch.where(x > lo + box, x - box, x)
            x = torch.where(x < lo, x + box, x)
        parts.append(x)
    x = torch.cat(parts)
    out = {"xyz": x}
    if kind in ("plain", "chains"):
        if case.get("rdf_bins"):
            out["counts"] = None
    else:
        out["types"] = None
    return out
