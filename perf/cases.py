"""The work that users of this framework have it do, as timed cases.

A case is one of five kinds of program:

  step    a `data` dictionary (structure and neighbour list) is in hand and the model is called on it: what the
          conversion tool times, what a training-set evaluation or a driver with its own neighbour list does
  fresh   a structure nobody has a list for: neighbour search, then the model (screening, or the pair style of a
          domain-decomposed MD code, which builds everything anew at every call; `ghosts` is the share of atoms owned
          by other ranks and takes the LAMMPS wrapper)
  md      a stretch of molecular dynamics through DeviceCalculator, everything on the GPU, list rebuilds included
  ase     the same through the ASE calculator protocol: positions come from the host, energy, forces and stress go back
  layer   one interaction layer put together from the op modules under autograd, forward and backward, in fp32 or fp64:
          what a model other than the one shipped here does with `cuda_mace.ops`
"""
import math
import os
import sys
from collections import OrderedDict

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "cuda-mace_amd"))

from cuda_mace.calculators import DeviceCalculator, LAMMPS_MACE, MACECalculator  # noqa: E402
from cuda_mace.models import OptimizedInvariantMACE, SyntheticInvariantMACE  # noqa: E402
from cuda_mace.ops import CubicSpline, InvariantMessagePassingTP, Linear, SymmetricContraction  # noqa: E402
from cuda_mace.ops.spherical_harmonics import SphericalHarmonics  # noqa: E402
from cuda_mace.utils.neighbour_list import neighbour_data  # noqa: E402

DEV = "cuda"
CUTOFF = 5.0
MD_STEPS = 24
ASE_STEPS = 8
PERIODIC = (True, True, True)
BALL = 4.0 / 3.0 * math.pi * CUTOFF ** 3


def listed():
    def case(name, kind, atoms, channels, **more):
        base = {"name": name, "kind": kind, "atoms": atoms, "channels": channels, "graphs": 1, "elements": 10, "density": 0.1,
                "periodic": True, "want": "forces", "ghosts": 0.0, "degree": 0, "dtype": "f32", "mixing": "shared"}
        base.update(more)
        return base

    return [
        # one small molecule, the smallest call: 21 atoms of {H, C, N, O} in vacuum
        case("molecule", "step", 21, 64, elements=4, density=0.041, periodic=False),
        # many such molecules per call: evaluation of a data set, serving
        case("molecules x512", "step", 21, 64, elements=4, density=0.041, graphs=512, periodic=False),
        # the conversion tool's benchmark crystal (216 atoms of carbon at diamond's density), relaxed or run by an ASE script
        case("ase crystal", "ase", 216, 128, elements=1, density=0.176, want="stress"),
        # constant-pressure work on an ordinary box: forces and stress
        case("box stress", "step", 5000, 96, want="stress"),
        # the headline workload
        case("box forces", "step", 25000, 128),
        # the largest box in ordinary use on one GPU, wide features
        case("large box forces", "step", 100000, 192),
        # energies alone: Monte Carlo moves, committee screening; a width that is no power of two
        case("energy", "step", 10007, 160, elements=4, want="energy"),
        # a structure without a list
        case("fresh structure", "fresh", 2000, 128, elements=4),
        # one rank of a domain-decomposed run: local atoms and ghosts, virials
        case("ghosts", "fresh", 12000, 256, elements=4, periodic=False, ghosts=0.45, want="stress"),
        # molecular dynamics on the GPU
        case("md", "md", 25000, 128, want="forces"),
        # op modules at the shape of the stand-alone message-passing benchmark
        case("layer", "layer", 4096, 96, degree=30),
        # the same ops in double precision: reference values, finite-difference checks
        case("layer f64", "layer", 1000, 64, degree=30, dtype="f64", mixing="none"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Any of the programs above at any size, width, composition and density that they meet."""
    kind = rng.choice(["step", "step", "step", "step", "batch", "batch", "ase", "fresh", "fresh", "md", "layer", "layer"])
    channels = 32 * rng.choice([1, 2, 2, 3, 3, 4, 4, 4, 5, 6, 7, 8])
    case = {"kind": kind, "atoms": 0, "channels": channels, "graphs": 1, "elements": rng.choice([1, 2, 4, 10]),
            "density": round(rng.uniform(0.05, 0.12), 3), "periodic": rng.random() < 0.75, "want": "forces", "ghosts": 0.0,
            "degree": 0, "dtype": "f32", "mixing": "shared"}
    if kind == "step":
        case["atoms"] = _log_int(rng, 20, min(100000, 14_000_000 // channels))
        case["want"] = rng.choice(["forces", "forces", "stress", "energy"])
    elif kind == "batch":
        case["kind"] = "step"
        case["periodic"] = rng.random() < 0.3
        case["atoms"] = _log_int(rng, 8, 300)
        case["graphs"] = _log_int(rng, 2, 32 if case["periodic"] else max(2, min(600, 40000 // case["atoms"])))
    elif kind == "ase":
        case["atoms"] = _log_int(rng, 20, 3000)
        case["want"] = "stress" if case["periodic"] else "forces"
    elif kind == "fresh":
        case["atoms"] = _log_int(rng, 30, 30000)
        if rng.random() < 0.4:
            case["periodic"], case["ghosts"], case["want"] = False, round(rng.uniform(0.2, 0.7), 2), rng.choice(["forces", "stress"])
    elif kind == "md":
        case["atoms"] = _log_int(rng, 100, min(25000, 3_200_000 // channels))
    else:
        case["degree"] = rng.randint(8, 60)
        case["dtype"] = rng.choice(["f32", "f32", "f64"])
        case["mixing"] = rng.choice(["shared", "element"]) if case["dtype"] == "f32" else "none"
        room = 100_000_000 if case["dtype"] == "f32" else 10_000_000
        case["atoms"] = _log_int(rng, 100, min(20000, room // (case["degree"] * channels)))
    if case["want"] == "stress" and case["kind"] == "step":
        case["periodic"] = True
    return case


# ---- structures -------------------------------------------------------------------------------------------------------
def _positions(case, g):
    """[graphs, atoms, 3] fp64 and the edge length of their cubic boxes: random sites of a cubic lattice, each moved by up
    to 0.3 lattice spacings per axis (a dense disordered phase without close pairs)."""
    n, graphs = case["atoms"], case["graphs"]
    box = (n / case["density"]) ** (1.0 / 3.0)
    m = int(math.ceil(n ** (1.0 / 3.0) - 1e-9))
    if m ** 3 == n and n < 1000:
        m += 1  # leave some sites empty in the small ones too
    sites = torch.rand(graphs, m ** 3, generator=g).argsort(dim=1)[:, :n]
    grid = torch.stack([sites // (m * m), (sites // m) % m, sites % m], dim=-1).double()
    jitter = 0.6 * (torch.rand(graphs, n, 3, generator=g, dtype=torch.float64) - 0.5)
    return (grid + 0.5 + jitter) * (box / m), box


def _species(case, count, g):
    """Element index per atom; the k-th element is 1 / (k + 1) as common as the first."""
    weights = 1.0 / torch.arange(1, case["elements"] + 1, dtype=torch.float64)
    return torch.multinomial(weights, count, replacement=True, generator=g)


def _one_hot(case, count, g):
    return torch.nn.functional.one_hot(_species(case, count, g), case["elements"]).double()


def _neighbours_per_atom(case):
    if case["kind"] == "layer":
        return float(case["degree"])
    if case["periodic"]:
        return case["density"] * BALL
    # a cube without periodic images loses the part of the ball that sticks out (to first order in cutoff / box)
    box = (case["atoms"] / case["density"]) ** (1.0 / 3.0)
    return min(case["atoms"] - 1.0, case["density"] * BALL) * max(0.35, 1.0 - 9.0 * CUTOFF / (16.0 * box))


_MODELS = OrderedDict()  # a program has one model and many structures


def _model_of(case):
    key = (case["channels"], case["elements"])
    if key not in _MODELS:
        while len(_MODELS) >= 2:
            _MODELS.popitem(last=False)
        up = SyntheticInvariantMACE(channels=case["channels"], atomic_numbers=tuple(range(1, case["elements"] + 1)),
                                    avg_num_neighbors=40.0, seed=0)
        _MODELS[key] = (up, OptimizedInvariantMACE(up, device=DEV))
    return _MODELS[key]


class _Atoms:
    """The four accessors of ase.Atoms that the calculator reads."""

    def __init__(self, positions, numbers, cell, pbc):
        self.positions, self.numbers, self.cell, self.pbc = positions, numbers, cell, pbc

    def get_positions(self):
        return self.positions

    def get_atomic_numbers(self):
        return self.numbers

    def get_cell(self):
        return self.cell

    def get_pbc(self):
        return self.pbc


def _trajectory(positions, steps, g):
    """`steps` frames that lead from `positions` away and back: thermal directions, the fastest atom 0.4 A out and back, so
    that a list with a skin of 0.5 A is rebuilt about once in ten to twelve steps."""
    v = torch.randn(positions.shape, generator=g, dtype=torch.float64)
    v = v * (0.4 / float(v.norm(dim=1).max()))
    phase = [0.5 - 0.5 * math.cos(2.0 * math.pi * k / steps) for k in range(steps)]
    return [positions + p * v for p in phase]


def _batch(case, g):
    """The data dictionary of `graphs` structures, collated as a data loader does."""
    pos, box = _positions(case, g)
    graphs, n = pos.shape[0], pos.shape[1]
    attrs = _one_hot(case, graphs * n, g).to(DEV)
    pos = pos.to(DEV)
    cell = torch.eye(3, dtype=torch.float64, device=DEV) * box
    if case["periodic"]:
        parts = [neighbour_data(pos[k], attrs[:1], CUTOFF, PERIODIC, cell) for k in range(graphs)]
        data = {"edge_index": torch.cat([p["edge_index"] + k * n for k, p in enumerate(parts)], dim=1).contiguous(),
                "shifts": torch.cat([p["shifts"] for p in parts]), "unit_shifts": torch.cat([p["unit_shifts"] for p in parts]),
                "cell": cell.repeat(graphs, 1)}
    else:
        apart = torch.arange(graphs, device=DEV, dtype=torch.float64).view(-1, 1, 1) * (box + 4.0 * CUTOFF)
        spread = (pos + torch.cat([apart, torch.zeros_like(apart), torch.zeros_like(apart)], dim=-1)).reshape(-1, 3)
        part = neighbour_data(spread, attrs, CUTOFF)
        data = {"edge_index": part["edge_index"].clone(), "shifts": part["shifts"], "unit_shifts": part["unit_shifts"],
                "cell": torch.zeros(3 * graphs, 3, dtype=torch.float64, device=DEV)}
    data.update(positions=pos.reshape(-1, 3).contiguous(), node_attrs=attrs,
                batch=torch.arange(graphs, device=DEV).repeat_interleave(n),
                ptr=torch.arange(graphs + 1, device=DEV) * n)
    return data


def _layer(case, g):
    n, degree, c = case["atoms"], case["degree"], case["channels"]
    dtype = torch.float64 if case["dtype"] == "f64" else torch.float32
    up, model = _model_of(case)
    edges = n * degree  # the degrees of single nodes vary about their mean
    receiver = torch.randint(0, n, (edges,), generator=g).sort().values
    sender = torch.randint(0, n, (edges,), generator=g)
    # lengths as a disordered phase has them: uniform over the ball beyond the shortest bond
    length = (torch.rand(edges, 1, generator=g, dtype=torch.float64) * (CUTOFF ** 3 - 1.0) + 1.0) ** (1.0 / 3.0)
    direction = torch.randn(edges, 3, generator=g, dtype=torch.float64)
    vectors = direction / direction.norm(dim=1, keepdim=True) * length
    knots = torch.linspace(1e-12, CUTOFF + 1.0, 256, dtype=torch.float64)
    with torch.no_grad():
        radial = up.radial_embedding(knots.unsqueeze(-1), None, None, None)
        table = up.interactions[0].conv_tp_weights(radial[0] if isinstance(radial, tuple) else radial)
    spline = CubicSpline(knots.to(dtype), table.to(dtype), float(knots[1] - knots[0]), CUTOFF).to(DEV)
    linear = {"shared": lambda: Linear(up.interactions[1].linear).to(DEV), "element": lambda: model.interactions[0].skip_tp,
              "none": lambda: None}[case["mixing"]]()
    one_hot = _one_hot(case, n, g).float().to(DEV)
    return {
        "kind": "layer", "harmonics": SphericalHarmonics(), "spline": spline, "tp": InvariantMessagePassingTP(), "linear": linear,
        "contraction": SymmetricContraction(up.products[1].symmetric_contractions, device=DEV, dtype=dtype),
        "one_hot": one_hot if case["mixing"] == "element" else None, "types": one_hot.argmax(dim=1).int(),
        "vectors": vectors.to(DEV, dtype).requires_grad_(True), "sender": sender.int().to(DEV), "receiver": receiver.int().to(DEV),
        "feats": torch.randn(n, c, generator=g, dtype=torch.float64).to(DEV, dtype).requires_grad_(True),
        "seed": torch.randn(n, 1, c, generator=g, dtype=torch.float64).to(DEV, dtype), "nodes": n,
    }


def prepare(case, seed):
    g = torch.Generator().manual_seed(int(seed))
    kind = case["kind"]
    if kind == "layer":
        return _layer(case, g)
    model = _model_of(case)[1]
    state = {"kind": kind, "model": model, "want": case["want"]}
    if kind == "step":
        state["data"] = _batch(case, g)
        return state
    pos, box = _positions(case, g)
    pos, n = pos[0], case["atoms"]
    pbc = PERIODIC if case["periodic"] else (False, False, False)
    cell = torch.eye(3, dtype=torch.float64) * box
    if kind == "ase":
        numbers = _species(case, n, g).numpy() + 1
        state["frames"] = [_Atoms(p.numpy().copy(), numbers, cell.numpy() if case["periodic"] else np.zeros((3, 3)), pbc)
                           for p in _trajectory(pos, ASE_STEPS, g)]
        state["calc"] = MACECalculator(model, device=DEV)
        state["properties"] = ["energy", "forces"] + (["stress"] if case["want"] == "stress" else [])
        return state
    attrs = _one_hot(case, n, g).to(DEV)
    cell = cell.to(DEV) if case["periodic"] else None
    if kind == "md":
        state["frames"] = [p.to(DEV) for p in _trajectory(pos, MD_STEPS, g)]
        state["calc"] = DeviceCalculator(model, attrs, cutoff=CUTOFF, skin=0.5, pbc=pbc, cell=cell)
        return state
    state.update(positions=pos.to(DEV), attrs=attrs, pbc=pbc, cell=cell, local=None)
    if case["ghosts"] > 0.0:
        state["local"] = (pos[:, 0] < (1.0 - case["ghosts"]) * box).to(DEV)
        state["wrapper"] = LAMMPS_MACE(model)
    return state


def _kept(out):
    return {k: v for k, v in out.items() if torch.is_tensor(v) and k != "displacement"}


def run(state):
    kind = state["kind"]
    if kind == "layer":
        feats, vectors = state["feats"], state["vectors"]
        lengths = vectors.norm(dim=1)
        harmonics = state["harmonics"](vectors)
        radial = state["spline"](lengths).view(lengths.numel(), 4, feats.shape[1])
        message = state["tp"](feats, harmonics, radial, state["sender"], state["receiver"], state["nodes"])
        if state["one_hot"] is not None:
            message = state["linear"](message, state["one_hot"])
        elif state["linear"] is not None:
            message = state["linear"](message)
        out = state["contraction"](message, state["types"])
        g_feats, g_vectors = torch.autograd.grad([out], [feats, vectors], [state["seed"]])
        return {"out": out.detach(), "g_feats": g_feats, "g_vectors": g_vectors}
    if kind == "step":
        if state["want"] == "energy":
            with torch.no_grad():
                return _kept(state["model"](dict(state["data"]), compute_force=False))
        return _kept(state["model"](dict(state["data"]), compute_stress=state["want"] == "stress"))
    if kind == "fresh":
        data = neighbour_data(state["positions"], state["attrs"], CUTOFF, state["pbc"], state["cell"])
        if state["local"] is not None:
            return _kept(state["wrapper"](data, state["local"], compute_virials=state["want"] == "stress"))
        return _kept(state["model"](data, compute_stress=state["want"] == "stress"))
    if kind == "md":
        outs = [state["calc"].compute(p) for p in state["frames"]]
        return {"energy": [o["energy"] for o in outs], "forces": [o["forces"] for o in outs]}
    results = []
    for atoms in state["frames"]:
        state["calc"].calculate(atoms, state["properties"])
        results.append(state["calc"].results)
    return [{k: r[k] for k in state["properties"]} for r in results]


def work(case):
    n, c = case["atoms"] * case["graphs"], case["channels"]
    e = n * _neighbours_per_atom(case)
    if case["kind"] == "layer":
        s = 8 if case["dtype"] == "f64" else 4
        mix = 0 if case["mixing"] == "none" else 2 * 2 * 16 * n * c * c
        # forward: cubic of 4 degrees, products, 16 accumulations per edge and channel; backward: twice that; contraction
        return {"bytes": s * (2 * n * c + 2 * n * c + 2 * 3 * e + 16 * 4 * c * 255) + 8 * e, "flops": 3 * 60 * e * c + mix + 800 * n * c}
    forward = 2 * 60 * e * c + 2 * (2 * 16 * n * c * c) + 2 * 400 * n * c + 8 * n * c * c
    backward = 2 * 120 * e * c + 2 * (2 * 16 * n * c * c) + 8 * n * c * c
    flops = forward + (0 if case["want"] == "energy" else backward)
    weights = 4 * (2 * 255 * 16 * c + case["elements"] * 5 * c * c + 8 * c * c)
    arrays = 24 * n + 8 * case["elements"] * n + (0 if case["want"] == "energy" else 24 * n) + 8 * n
    feats = 16 * n * c
    lists = 8 * e + (24 * e if case["periodic"] else 0)  # two indices and, between images, a shift per pair
    steps = {"md": MD_STEPS, "ase": ASE_STEPS}.get(case["kind"], 1)
    if case["kind"] == "step":
        return {"bytes": arrays + feats + lists + weights, "flops": flops}
    if case["kind"] == "fresh":
        return {"bytes": arrays + feats + weights, "flops": flops}
    return {"bytes": steps * (arrays + weights), "flops": steps * flops}


def tolerance(case):
    if case["dtype"] == "f64":
        return {"rel": 1e-12}
    # fp32 sums of a few hundred terms, features and gradients through two layers; single components lose digits to
    # cancellation
    return {"rel": 1e-5, "max": 1e-3}
