"""Performance cases of the MD framework: what its users run, through its public entry points.

Kinds of case (``case["kind"]``):

* ``md``        a short NVT Nose-Hoover run in whole-step mode from a stored state (``model``
                "mace": 2 layers, ``channels`` wide; "threebody": 4 layers, bonds to ``bond_cutoff``);
* ``evaluate``  energy and forces at host coordinates (a relaxation, a path search, an MD driver of
                the caller's own), candidates kept between the calls;
* ``ragged``    the exact ragged neighbour list of new coordinates (eager MD and the model-graph mode);
* ``fixed``     the fixed-capacity neighbour list, candidates refreshed and edges rebuilt, optionally
                with the three-body line graph;
* ``segment``   the receiver sum of edge rows and its VJP, on the neighbour list's own CSR;
* ``gather``    the edge rows [edge | sender | receiver] of a model and their VJP, from plain indices;
* ``linear``    the wide edge projection in float32 and its input gradient;
* ``gemm16``    the same projection on bf16 operands;
* ``fourier``   the angle basis of the triplets and its VJP;
* ``block``     one edge block as a model composes it: edge rows -> projection -> weighted receiver sum,
                forward and backward.

Systems are ABX3 perovskite supercells (5 atoms per 6.2 A cell) with thermal displacements, cut off at
6 A; features are standard normal, weights scaled by their fan-in. The reference values of ``exact`` are
plain torch in float64 on pair lists formed here.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from fastmd_amd.config import InferenceConfig
from fastmd_amd.execution.skin_topology import SkinTopologyRunner
from fastmd_amd.graph.fixed_capacity_builder import FixedCapacityGraphBuilder
from fastmd_amd.graph.gpu_graph_builder import TensorGraphBuilder
from fastmd_amd.adapters.protocol import PaddingRule
from fastmd_amd.interfaces.gpu_md import GPUResidentMolecularDynamics
from fastmd_amd.models.mace_like import MaceLike, MaceLikeAdapter, MaceLikeConfig
from fastmd_amd.models.threebody_like import ThreeBodyAdapter, ThreeBodyConfig, ThreeBodyLike
from fastmd_amd.ops.csr_segment_sum import csr_segment_sum
from fastmd_amd.ops.gather_cat import aligned_gather_cat3
from fastmd_amd.ops.segment import weighted_segment_sum
from fastmd_amd.ops.threebody import threebody_fourier_basis
from fastmd_amd.ops.wide_gemm import gemm, linear
from fastmd_amd.systems import System

DEVICE = "cuda"
LATTICE = 6.2
CUTOFF = 6.0
N_BASIS = 8
ELEMENTS = (55, 50, 53)
MASSES = {55: 133.0, 50: 119.0, 53: 127.0}
KB = 1.38064852e-23 / 1.6021766208e-19  # eV / K
FS = 1e-5 * math.sqrt(1.6021766208e-19 / 1.660539040e-27)  # one fs in A sqrt(amu / eV)
TEMPERATURE, TIMESTEP, TDAMP, TCHAIN = 500.0, 0.25, 25.0, 3
STEPS_PER_LAUNCH = 10
SHEAR = 0.1  # of the second and third lattice vector, for triclinic cells
# of the about 16.7 edges per atom, and of the bonds and ordered bond pairs per atom below a line-graph
# cutoff, what the operator cases keep
EDGES_PER_ATOM = 16
FOURIER_ROWS = {3.5: (1.8, 3.0), 4.0: (3.0, 7.0), 4.5: (7.2, 42.0)}


# ---------------------------------------------------------------------------------------- cases


def listed():
    return [
        # the published protocol's system size: every launch and every dependent step counts
        _md("md_mace_135", "mace", (3, 3, 3), 128, 40),
        # the headline system
        _md("md_mace_10000", "mace", (10, 10, 20), 128, 20),
        # a bond-angle model: line graph, Fourier angles, angle -> bond -> atom sums every step
        _md("md_threebody_5000", "threebody", (10, 10, 10), 64, 20, bond_cutoff=3.5),
        # single points driven from the host (optimizers, path searches)
        {"name": "evaluate_mace_1080", "kind": "evaluate", "model": "mace", "nx": 6, "ny": 6, "nz": 6, "channels": 64,
         "bond_cutoff": 0.0},
        # the neighbour list of eager MD at an odd supercell, and of a large whole-step system's refresh
        {"name": "ragged_3430", "kind": "ragged", "nx": 7, "ny": 7, "nz": 14, "shear": 0.0},
        {"name": "fixed_40000", "kind": "fixed", "nx": 20, "ny": 20, "nz": 20, "shear": 0.0, "line_cutoff": 0.0},
        # the operators at the sizes of the operator benchmark
        {"name": "segment_40000_f128", "kind": "segment", "nx": 20, "ny": 20, "nz": 20, "F": 128, "weighted": False},
        {"name": "gather_10000_f128", "kind": "gather", "nx": 10, "ny": 10, "nz": 20, "F": 128},
        {"name": "linear_10000_f256", "kind": "linear", "nx": 10, "ny": 10, "nz": 20, "F": 256, "bias": True},
        {"name": "gemm16_40000_f128", "kind": "gemm16", "nx": 20, "ny": 20, "nz": 20, "F": 128},
        # the angle basis at the size of a line graph at 4.5 A, the default bond cutoff
        {"name": "fourier_2560", "kind": "fourier", "nx": 8, "ny": 8, "nz": 8, "line_cutoff": 4.5, "n_freq": 4},
        # the smallest call: one block of a small molecule crystal, forward and backward
        {"name": "block_135_f64", "kind": "block", "nx": 3, "ny": 3, "nz": 3, "F": 64},
    ]


def _md(name, model, cells, channels, steps, bond_cutoff=0.0):
    return {"name": name, "kind": "md", "model": model, "nx": cells[0], "ny": cells[1], "nz": cells[2],
            "channels": channels, "steps": steps, "bond_cutoff": bond_cutoff}


def draw(rng):
    kind = rng.choice(["md", "md", "evaluate", "ragged", "fixed", "segment", "gather", "linear", "gemm16", "fourier",
                       "block"])
    most = {"md": 2000, "evaluate": 2000, "block": 1000, "fourier": 512, "linear": 2000}.get(kind, 8000)
    case = {"kind": kind}
    if kind in ("md", "evaluate"):
        case["model"] = rng.choice(["mace", "mace", "threebody"])
        if case["model"] == "threebody":
            most, case["bond_cutoff"], case["channels"] = 800, rng.choice([3.0, 3.5]), rng.choice([64, 128])
            most = most * 64 // case["channels"]
        else:
            case["bond_cutoff"], case["channels"] = 0.0, rng.choice([64, 128, 256])
            most = most * 128 // max(128, case["channels"])
    cells = math.exp(rng.uniform(math.log(27.0), math.log(most)))
    nx, ny = (max(3, round(cells ** (1 / 3) * math.exp(rng.uniform(-0.25, 0.25)))) for _ in range(2))
    nz = max(3, round(cells / (nx * ny)))
    while nx * ny * nz > most and max(nx, ny, nz) > 3:
        nx, ny, nz = (n - 1 if n == max(nx, ny, nz) else n for n in (nx, ny, nz))
    case.update(nx=nx, ny=ny, nz=nz)
    if kind == "md":
        case["steps"] = 40 if case["model"] == "mace" and nx * ny * nz <= 100 else 20
    elif kind == "ragged":
        case["shear"] = rng.choice([0.0, SHEAR])
    elif kind == "fixed":
        case.update(shear=rng.choice([0.0, SHEAR]), line_cutoff=rng.choice([0.0, 3.0, 3.5]))
    elif kind == "segment":
        case.update(F=rng.choice([64, 100, 128, 250, 256]), weighted=rng.choice([False, True]))
    elif kind == "gather":
        case["F"] = rng.choice([64, 100, 128, 250, 256])
    elif kind == "linear":
        case.update(F=rng.choice([64, 100, 128, 256]), bias=rng.choice([False, True]))
    elif kind == "gemm16":
        case["F"] = rng.choice([64, 100, 128])
    elif kind == "fourier":
        case.update(line_cutoff=rng.choice([3.5, 4.0, 4.5]), n_freq=rng.choice([3, 4, 5]))
    elif kind == "block":
        case["F"] = rng.choice([64, 100, 128])
    return case


def _atoms(case):
    return 5 * case["nx"] * case["ny"] * case["nz"]


# ---------------------------------------------------------------------------------------- inputs


def _system(case, seed):
    """Positions [N, 3] float64, cell [3, 3], numbers [N] of the displaced supercell."""
    repeats = np.array([case["nx"], case["ny"], case["nz"]])
    sites = np.array([[0.0, 0.0, 0.0], [0.5, 0.5, 0.5], [0.5, 0.5, 0.0], [0.5, 0.0, 0.5], [0.0, 0.5, 0.5]])
    grid = np.stack(np.meshgrid(*[np.arange(k) for k in repeats], indexing="ij"), -1).reshape(-1, 3)
    frac = (grid[:, None, :] + sites[None]).reshape(-1, 3) / repeats
    cell = np.diag(repeats * LATTICE)
    if case.get("shear"):
        cell[1, 0] = case["shear"] * cell[1, 1]
        cell[2, 1] = case["shear"] * cell[2, 2]
    rng = np.random.default_rng(seed)
    # 0.25 A: thermal motion at some hundred K. The ragged list's length is that of its edges, which stays
    # the same from seed to seed in a crystal near rest: no shell of the lattice lies within 0.2 A of the cutoff
    positions = frac @ cell + rng.normal(0.0, 0.02 if case["kind"] == "ragged" else 0.25, frac.shape)
    numbers = np.tile(np.array([55, 50, 53, 53, 53], dtype=np.int32), int(np.prod(repeats)))
    return positions, cell, numbers


def _momenta(numbers, seed):
    m = np.array([MASSES[int(z)] for z in numbers])
    rng = np.random.default_rng(seed + 7919)
    return rng.standard_normal((len(m), 3)) * np.sqrt(m * KB * TEMPERATURE)[:, None], m


def _weights(case, seed):
    """A model's parameters (a checkpoint, as the program would load it), float32 on the CPU."""
    C, gen = case["channels"], torch.Generator().manual_seed(seed)

    def rnd(*shape, fan_in=1):
        return torch.randn(*shape, generator=gen) / math.sqrt(fan_in)

    w = {"embedding": rnd(3, C), "e0": -1.0 - torch.rand(3, generator=gen)}
    if case["model"] == "mace":
        for t in range(2):
            p = f"layers.{t}."
            w[p + "W1"] = rnd(2 * C + N_BASIS, 4 * C, fan_in=2 * C + N_BASIS)
            for name in ("Wm0", "Wm1", "Wo0", "Wo1", "Wsc0"):
                w[p + name] = rnd(C, C, fan_in=C)
            w[p + "Wc"], w[p + "Wd"] = rnd(3, 5, C, fan_in=5), rnd(3, 4, C, fan_in=4)
        w["wr1"], w["Wr2a"], w["wr2b"] = rnd(C, fan_in=C), rnd(C, 16, fan_in=C), rnd(16, fan_in=16)
    else:
        w["We"] = rnd(N_BASIS, C, fan_in=N_BASIS)
        for t in range(4):
            w[f"layers.{t}.W3"] = rnd(3 * C + 9, C, fan_in=3 * C + 9)
            w[f"layers.{t}.W2"] = rnd(3 * C, C, fan_in=3 * C)
        w["wr"] = rnd(C, fan_in=C)
    return w


def _adapter(case, seed):
    if case["model"] == "mace":
        module, wrap = MaceLike(MaceLikeConfig(channels=case["channels"])), MaceLikeAdapter
    else:
        module = ThreeBodyLike(ThreeBodyConfig(channels=case["channels"], bond_cutoff=case["bond_cutoff"]))
        wrap = ThreeBodyAdapter
    module.load_state_dict(_weights(case, seed), strict=False)
    return wrap(module, device=DEVICE)


def _pairs(positions, lengths, cutoff):
    """(centre, neighbour, image) of every pair below ``cutoff`` in an orthorhombic cell of at least
    twice the cutoff, rows by centre then neighbour; plain torch, float64."""
    n = positions.shape[0]
    step = max(1, 20_000_000 // n)
    out = []
    for a in range(0, n, step):
        d = positions[None, :, :] - positions[a:a + step, None, :]
        image = -torch.round(d / lengths)
        r2 = ((d + image * lengths) ** 2).sum(2)
        r2[torch.arange(d.shape[0], device=d.device), torch.arange(a, a + d.shape[0], device=d.device)] = 1e9
        i, j = torch.nonzero(r2 < cutoff * cutoff, as_tuple=True)
        out.append((i + a, j, image[i, j]))
        del d, image, r2
    return tuple(torch.cat(part) for part in zip(*out))


def _edges(case, seed, cutoff=CUTOFF):
    """The pair list of the case's system on the GPU: positions (wrapped), centre, neighbour, image."""
    positions, cell, _ = _system(case, seed)
    lengths = torch.tensor(np.diag(cell), device=DEVICE)
    q = torch.tensor(positions, device=DEVICE) % lengths
    return (q, *_pairs(q, lengths, cutoff))


def _cut(rows, count, seed):
    """``count`` of the rows, in their order (the operands of another seed have the same shapes)."""
    if rows < count:
        raise ValueError(f"{rows} rows of {count}")
    gen = torch.Generator(device=DEVICE).manual_seed(seed + 104729)
    return torch.randperm(rows, generator=gen, device=DEVICE)[:count].sort()[0]


def _offsets(index, n):
    off = torch.zeros(n + 1, dtype=torch.int64, device=index.device)
    off[1:] = torch.cumsum(torch.bincount(index, minlength=n), 0)
    return off


def _triplets(centre, n):
    """Every ordered pair (b1, b2) of two distinct rows of one centre (rows sorted by centre)."""
    count = torch.bincount(centre, minlength=n)
    first = torch.cumsum(count, 0) - count
    per_row = count[centre]
    b1 = torch.repeat_interleave(torch.arange(centre.numel(), device=centre.device), per_row)
    rank = torch.arange(b1.numel(), device=centre.device) - torch.repeat_interleave(torch.cumsum(per_row, 0) - per_row, per_row)
    b2 = first[centre[b1]] + rank
    keep = b1 != b2
    return b1[keep], b2[keep]


class _Random:
    """Standard normal tensors on the GPU, from a seed."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEVICE).manual_seed(seed)

    def __call__(self, *shape, fan_in=1, dtype=torch.float32):
        return (torch.randn(*shape, generator=self.gen, device=DEVICE) / math.sqrt(fan_in)).to(dtype)


def _tensors(case, seed):
    """The operands of an operator case (graph indices as int32, as the builders publish them)."""
    kind, n, F, rnd = case["kind"], _atoms(case), case.get("F", 0), _Random(seed)
    if kind == "fourier":
        q, c, j, image = _edges(case, seed, case["line_cutoff"])
        lengths = torch.tensor([case["nx"], case["ny"], case["nz"]], device=DEVICE, dtype=torch.float64) * LATTICE
        rows, triplets = FOURIER_ROWS[case["line_cutoff"]]
        keep = _cut(c.numel(), int(rows * n), seed)
        c, j, image = c[keep], j[keep], image[keep]
        v = q[j] + image * lengths - q[c]
        b1, b2 = _triplets(c, n)
        keep = _cut(b1.numel(), int(triplets * n), seed)
        b1, b2 = b1[keep], b2[keep]
        unit = (v / v.norm(dim=1, keepdim=True)).float()
        return {"unit": unit, "target": b1.int(), "source": b2.int(), "gout": rnd(b1.numel(), 1 + 2 * case["n_freq"]),
                "freqs": torch.arange(1, case["n_freq"] + 1, dtype=torch.float32, device=DEVICE)}
    _, c, j, _ = _edges(case, seed)
    e, k = EDGES_PER_ATOM * n, 2 * F + N_BASIS
    keep = _cut(c.numel(), e, seed)
    c, j = c[keep], j[keep]
    t = {"centre": c.int(), "neighbour": j.int(), "off": _offsets(c, n)}
    if kind == "segment":
        t.update(value=rnd(e, F), weight=rnd(e, F) if case["weighted"] else None, gout=rnd(n, F))
    elif kind == "gather":
        t.update(ef=rnd(e, N_BASIS), x=rnd(n, F), gout=rnd(e, k))
    elif kind == "linear":
        t.update(rows=rnd(e, k), w=rnd(4 * F, k, fan_in=k), bias=rnd(4 * F) if case["bias"] else None, gout=rnd(e, 4 * F))
    elif kind == "gemm16":
        t.update(rows=rnd(e, k, dtype=torch.bfloat16), w=rnd(4 * F, k, fan_in=k, dtype=torch.bfloat16))
    elif kind == "block":
        t.update(ef=rnd(e, N_BASIS), x=rnd(n, F), w=rnd(F, k, fan_in=k), gate=rnd(e, 1).sigmoid(), gout=rnd(n, F))
    return t


# ---------------------------------------------------------------------------------------- passes


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("md", "evaluate"):
        positions, cell, numbers = _system(case, seed)
        adapter = _adapter(case, seed)
        if kind == "evaluate":
            runner = SkinTopologyRunner(adapter, atomic_numbers=numbers, cell=cell, device=DEVICE)
            runner.evaluate(positions)  # the candidates and the captured bucket that a program keeps
            return {"kind": kind, "runner": runner, "positions": positions}
        momenta, masses = _momenta(numbers, seed)
        md = GPUResidentMolecularDynamics(System(positions, cell, numbers, masses), model=adapter, device=DEVICE,
                                          temperature=TEMPERATURE, timestep=TIMESTEP, tdamp=TDAMP, tchain=TCHAIN,
                                          momenta=momenta, config=InferenceConfig(execution="whole_step"),
                                          steps_per_launch=STEPS_PER_LAUNCH)
        return {"kind": kind, "md": md, "start": md.integrator.snapshot(), "steps": case["steps"]}
    if kind in ("ragged", "fixed"):
        positions, cell, numbers = _system(case, seed)
        args = dict(cell=torch.tensor(cell), atomic_numbers=torch.tensor(numbers), atom_graph_cutoff=CUTOFF, device=DEVICE)
        if kind == "ragged":
            builder = TensorGraphBuilder(line_graph_cutoff=None, check_isolated_atoms=False, **args)
        else:
            line = case["line_cutoff"]
            n = _atoms(case)
            builder = FixedCapacityGraphBuilder(u_capacity=10 * n, t_capacity=8 * n if line else 0,
                                                line_graph_cutoff=line or None, candidate_cutoff=CUTOFF + 2.0,
                                                padding=PaddingRule("far_self_loops"), **args)
        return {"kind": kind, "builder": builder, "positions": torch.tensor(positions, device=DEVICE),
                "line": bool(case.get("line_cutoff"))}
    t = _tensors(case, seed)
    t.update(kind=kind, n=_atoms(case))
    for name in ("value", "weight", "x", "rows", "unit", "ef"):
        if t.get(name) is not None and kind != "gemm16":
            t[name].requires_grad_(True)
    return t


def run(state):
    return _RUN[state["kind"]](state)


def _run_md(s):
    md = s["md"]
    md.integrator.load_snapshot(s["start"])
    md.run(s["steps"])
    th = md.integrator
    return {"positions": th.positions, "momenta": th.momenta, "forces": th.forces, "energy": th.potential_energy}


def _run_evaluate(s):
    out = s["runner"].evaluate(s["positions"])
    return {"energy": out["e"], "forces": out["f"]}


def _run_ragged(s):
    g = s["builder"].build(s["positions"])
    return {"positions": g.positions, "edge_index": g.edge_index, "edge_image": g.edge_image,
            "edge_offsets": g.edge_offsets, "edge_reverse": g.edge_reverse}


def _run_fixed(s):
    b = s["builder"]
    _, status = b.build(s["positions"])
    g = b.batch
    out = {"positions": g.positions, "edge_index": g.edge_index, "edge_image": g.edge_image,
           "edge_offsets": g.edge_offsets, "edge_reverse": g.edge_reverse, "distances": b.distances,
           "overflow": status.overflow, "isolated": status.isolated_atom_count}
    if s["line"]:
        out.update(d2u=g.pair_d2u, u2d=g.pair_u2d, triplets=g.triplets, triplet_count=status.triplet_count)
    return out


def _run_segment(s):
    inputs = [s["value"]] if s["weight"] is None else [s["value"], s["weight"]]
    out = csr_segment_sum(s["value"], s["centre"], s["n"], off=s["off"], identity_perm=True, weight=s["weight"])
    return [out.detach(), *torch.autograd.grad(out, inputs, s["gout"])]


def _run_gather(s):
    rows = aligned_gather_cat3(s["ef"], s["x"], s["neighbour"], s["centre"])
    return [rows.detach(), *torch.autograd.grad(rows, (s["ef"], s["x"]), s["gout"])]


def _run_linear(s):
    out = linear(s["rows"], s["w"], s["bias"])
    return [out.detach(), *torch.autograd.grad(out, (s["rows"],), s["gout"])]


def _run_gemm16(s):
    return gemm(s["rows"], s["w"], b_layout=0)


def _run_fourier(s):
    out = threebody_fourier_basis(s["unit"], s["target"], s["source"], s["freqs"], math.sqrt(math.pi))
    return [out.detach(), *torch.autograd.grad(out, (s["unit"],), s["gout"])]


def _run_block(s):
    rows = aligned_gather_cat3(s["ef"], s["x"], s["neighbour"], s["centre"])
    z = linear(rows, s["w"])
    out = weighted_segment_sum(s["gate"], z, s["centre"], s["n"])
    return [out.detach(), *torch.autograd.grad(out, (s["ef"], s["x"]), s["gout"])]


_RUN = {"md": _run_md, "evaluate": _run_evaluate, "ragged": _run_ragged, "fixed": _run_fixed, "segment": _run_segment,
        "gather": _run_gather, "linear": _run_linear, "gemm16": _run_gemm16, "fourier": _run_fourier,
        "block": _run_block}


# ---------------------------------------------------------------------------------------- work


def _model_flops(case, n, edges):
    """Floating-point operations of one energy and force evaluation (the backward as twice the
    forward's edge side and once its node side), receiver and sender projections formed per atom."""
    C = case["channels"]
    if case["model"] == "mace":
        edge = sum(2 * N_BASIS * nz + 6 * nz + 14 * C for nz in (2 * C, 4 * C))
        node = 2 * C * C * (4 + 5 + 8 + 4 + 1) + 40 * C
        return 3 * edges * edge + 2 * n * node
    bonds, triplets = (0.9 * n, 0.8 * n) if case["bond_cutoff"] < 3.25 else (2.1 * n, 5.1 * n)
    layer = edges * (2 * C * C + 8 * C) + n * 8 * C * C + bonds * 4 * C * C + triplets * (18 * C + 10 * C)
    return 3 * 4 * layer


def work(case):
    kind, n = case["kind"], _atoms(case)
    e, F = EDGES_PER_ATOM * n, case.get("F", 0)
    k = 2 * F + N_BASIS
    if kind == "md":  # state in and out once per step, forces and energies besides
        return {"bytes": case["steps"] * n * 220, "flops": case["steps"] * _model_flops(case, n, e)}
    if kind == "evaluate":
        return {"bytes": n * 36, "flops": _model_flops(case, n, e)}
    if kind == "ragged":
        return {"bytes": n * (24 + 12 + 8) + e * (8 + 12 + 4), "flops": 27 * 5 * n * 8}
    if kind == "fixed":
        rows = 20 * n  # the capacity: padding rows are written too
        line = n * 8 * 20 + rows * 4 + 10 * n * 4 if case["line_cutoff"] else 0
        return {"bytes": n * (24 + 12 + 8) + rows * (8 + 12 + 4 + 4) + line, "flops": 27 * 5 * n * 8}
    if kind == "segment":
        return {"bytes": 4 * F * (2 * e + 2 * n) + 8 * n + (4 * F * 2 * e if case["weighted"] else 0), "flops": 2 * e * F}
    if kind == "gather":
        return {"bytes": 4 * (e * (2 * k + 2 * N_BASIS + 2) + 2 * n * F), "flops": 2 * e * F}
    if kind == "linear":
        return {"bytes": 4 * (e * (2 * k + 8 * F) + 8 * F * k), "flops": 4 * e * k * 4 * F}
    if kind == "gemm16":
        return {"bytes": 2 * (e * k + 4 * F * k) + 4 * e * 4 * F, "flops": 2 * e * k * 4 * F}
    if kind == "fourier":
        rows, pairs = FOURIER_ROWS[case["line_cutoff"]]
        width = 1 + 2 * case["n_freq"]
        return {"bytes": n * (pairs * (8 + 8 * width) + rows * 24), "flops": n * pairs * (40 + 20 * width)}
    return {"bytes": 4 * (e * (2 * N_BASIS + 3) + n * 4 * F + F * k), "flops": e * F * (4 * k + 6)}


def tolerance(case):
    # measured against float64 on one MI355X: forces of a model 2e-6 to 1e-5 (most of it the rounding of the
    # coordinates), sums 7e-8, projections 6e-7, bf16 operands (rounded in float64 too) 9e-8, angles 3e-7
    return {"md": {"rel": 2e-5, "max": 2e-4}, "evaluate": {"rel": 2e-5, "max": 2e-4},
            "ragged": {"rel": 1e-6, "max": 1e-6}, "fixed": {"rel": 1e-6, "max": 1e-6},
            "segment": {"rel": 5e-7, "max": 1e-5}, "gather": {"rel": 5e-7, "max": 1e-5},
            "linear": {"rel": 2.5e-6, "max": 2.5e-5}, "gemm16": {"rel": 1e-6, "max": 1e-5},
            "fourier": {"rel": 1.5e-6, "max": 1e-4}, "block": {"rel": 2.5e-6, "max": 2.5e-5}}[case["kind"]]


# ---------------------------------------------------------------------------------------- float64


def exact(case, seed):
    kind = case["kind"]
    if case.get("shear"):
        return None
    if kind in ("md", "evaluate"):
        return _exact_model(case, seed)
    if kind in ("ragged", "fixed"):
        q, c, j, image = _edges(case, seed)
        # the coordinates as published (the wrapped positions), the images only of an exact-size list
        return {"positions": q, "edge_index": None, "edge_image": image if kind == "ragged" else None,
                "edge_offsets": None, "edge_reverse": None}
    t = {k: v.double() if torch.is_tensor(v) and v.is_floating_point() else v for k, v in _tensors(case, seed).items()}
    for name in ("value", "weight", "x", "rows", "unit", "ef"):
        if t.get(name) is not None and kind != "gemm16":
            t[name].requires_grad_(True)
    n, F = _atoms(case), case.get("F", 0)
    if kind == "segment":
        rows = t["value"] if t["weight"] is None else t["value"] * t["weight"]
        out = _sum(rows, t["centre"].long(), n)
        inputs = [t["value"]] if t["weight"] is None else [t["value"], t["weight"]]
    elif kind == "gather":
        out, inputs = _rows(t), [t["ef"], t["x"]]
    elif kind == "linear":
        out, inputs = t["rows"] @ t["w"].t(), [t["rows"]]
        if t["bias"] is not None:
            out = out + t["bias"]
    elif kind == "gemm16":
        return t["rows"] @ t["w"].t()
    elif kind == "fourier":
        u = t["unit"]
        cosine = (u[t["target"].long()] * u[t["source"].long()]).sum(1) * (1 - 1e-6)
        out, inputs = _angles(cosine, case["n_freq"]), [u]
    else:
        out, inputs = _sum((_rows(t) @ t["w"].t()) * t["gate"], t["centre"].long(), n), [t["ef"], t["x"]]
    return [out.detach(), *torch.autograd.grad(out, inputs, t["gout"])]


def _sum(rows, index, n):
    return torch.zeros(n, *rows.shape[1:], dtype=rows.dtype, device=rows.device).index_add(0, index, rows)


def _rows(t):
    return torch.cat([t["ef"], t["x"][t["neighbour"].long()], t["x"][t["centre"].long()]], 1)


def _angles(cosine, n_freq):
    theta = torch.arccos(cosine)
    ph = theta[:, None] * torch.arange(1, n_freq + 1, dtype=theta.dtype, device=theta.device)
    return torch.cat([torch.full_like(theta[:, None], 2 ** -0.5), torch.sin(ph), torch.cos(ph)], 1) / math.sqrt(math.pi)


def _envelope(r, cutoff):
    x = r / cutoff
    return torch.where(x < 1, 1 - 21 * x ** 5 + 35 * x ** 6 - 15 * x ** 7, torch.zeros_like(x))


def _node_energy(case, p, q, lengths, elem, c, j, image):
    n = q.shape[0]
    v = q[j] + image * lengths - q[c]
    r = v.norm(dim=1)
    u, fc = v / r[:, None], _envelope(r, CUTOFF)
    k = torch.arange(1, N_BASIS + 1, dtype=q.dtype, device=q.device)
    ef = math.sqrt(2.0 / CUTOFF) * torch.sin(k * math.pi * r[:, None] / CUTOFF) / r[:, None] * fc[:, None]
    h = p["embedding"][elem]
    silu = torch.nn.functional.silu
    if case["model"] == "threebody":
        rb = case["bond_cutoff"]
        bonds = torch.nonzero(r.detach() < rb).flatten()
        s = _envelope(r, rb)
        t1, t2 = _triplets(c[bonds], n)
        b1, b2 = bonds[t1], bonds[t2]
        alpha = _angles((u[b1] * u[b2]).sum(1) * (1 - 1e-6), 4)
        eps = ef @ p["We"]
        for t in range(4):
            z3 = torch.cat([eps[b1], eps[b2], h[c[b1]], alpha], 1) @ p[f"layers.{t}.W3"]
            eps = eps.index_add(0, b1, silu(z3) * (s[b1] * s[b2])[:, None] / 4.0)
            z2 = torch.cat([h[j], h[c], eps], 1) @ p[f"layers.{t}.W2"]
            h = h.index_add(0, c, silu(z2) * fc[:, None] / 15.0)
        return p["e0"][elem] + h @ p["wr"]
    C = case["channels"]
    h1 = torch.zeros(n, 3, C, dtype=q.dtype, device=q.device)
    first = None
    for t in range(2):
        w = {name.split(".")[2]: x for name, x in p.items() if name.startswith(f"layers.{t}.")}
        z = torch.cat([h[j], h[c], ef], 1) @ w["W1"]
        wa, wb, wc, wd = (silu(z) * fc[:, None]).split(C, 1)
        m0 = wa * h[j] + wc * (h1[j] * u[:, :, None]).sum(1)
        m1 = (wb * h[j])[:, None, :] * u[:, :, None] + wd[:, None, :] * h1[j]
        P0, P1 = _sum(m0, c, n) / 15.0 @ w["Wm0"], _sum(m1, c, n) / 15.0 @ w["Wm1"]
        n1, a, d = (P1 * P1).sum(1), w["Wc"][elem], w["Wd"][elem]
        B0 = a[:, 0] * P0 + a[:, 1] * P0 ** 2 + a[:, 2] * n1 + a[:, 3] * P0 ** 3 + a[:, 4] * P0 * n1
        h1 = ((d[:, 0] + d[:, 1] * P0 + d[:, 2] * P0 ** 2 + d[:, 3] * n1)[:, None, :] * P1) @ w["Wo1"]
        h = B0 @ w["Wo0"] + h @ w["Wsc0"]
        first = h if first is None else first
    return p["e0"][elem] + first @ p["wr1"] + silu(h @ p["Wr2a"]) @ p["wr2b"]


def _exact_model(case, seed):
    positions, cell, numbers = _system(case, seed)
    lengths = torch.tensor(np.diag(cell), device=DEVICE)
    params = {k: v.double().to(DEVICE) for k, v in _weights(case, seed).items()}
    elem = torch.tensor([ELEMENTS.index(int(z)) for z in numbers], device=DEVICE)

    def forces(q):
        q = (q % lengths).detach()
        c, j, image = _pairs(q, lengths, CUTOFF)
        leaf = q.requires_grad_(True)
        energy = _node_energy(case, params, leaf, lengths, elem, c, j, image).sum()
        return energy.detach(), -torch.autograd.grad(energy, leaf)[0]

    q = torch.tensor(positions, device=DEVICE)
    energy, f = forces(q)
    if case["kind"] == "evaluate":
        return {"energy": energy, "forces": f}
    momenta, masses = _momenta(numbers, seed)
    p, m = torch.tensor(momenta, device=DEVICE), torch.tensor(masses, device=DEVICE)[:, None]
    n, dt, kT = len(masses), TIMESTEP * FS, KB * TEMPERATURE
    Q = [3 * n * kT * (TDAMP * FS) ** 2] + [kT * (TDAMP * FS) ** 2] * (TCHAIN - 1)
    w = 1 / (2 - 2 ** (1 / 3))
    pe = [0.0] * TCHAIN

    def kinetic2():
        return float((p * p / m).sum())

    def chain(i, ke2, delta):
        scale = math.exp(-pe[i + 1] * delta / 4 / Q[i + 1]) if i < TCHAIN - 1 else 1.0
        g = ke2 - 3 * n * kT if i == 0 else pe[i - 1] ** 2 / Q[i - 1] - kT
        pe[i] = (pe[i] * scale + g * delta / 2) * scale

    def thermostat():
        nonlocal p
        ke2 = kinetic2()
        for coeff in (w, -(2 ** (1 / 3)) * w, w):
            delta = coeff * dt / 2
            for i in reversed(range(TCHAIN)):
                chain(i, ke2, delta)
            p = p * math.exp(-delta * pe[0] / Q[0])
            ke2 = kinetic2()
            for i in range(TCHAIN):
                chain(i, ke2, delta)

    for _ in range(case["steps"]):
        thermostat()
        p = p + dt / 2 * f
        q = q + dt * p / m
        energy, f = forces(q)
        p = p + dt / 2 * f
        thermostat()
    return {"positions": q, "momenta": p, "forces": f, "energy": energy.reshape(1)}
