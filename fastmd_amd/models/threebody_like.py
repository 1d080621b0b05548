"""A CHGNet/MatRIS-style three-body interatomic potential whose forward and VJP run as HIP kernels.

The reference's three-body models are upstream CHGNet (wrapped by fastmd/models/chgnet.py:1-60,
356-366) and MatRIS (fastmd/models/matris/model.py, interaction_block.py); neither's weights nor
the upstream chgnet package are available here, so this package defines its own configs[4] model
"64 channels, 4 layers, atom graph 6 A, bond graph 3 A, angles expanded in Fourier terms" with
the reference's data path: the line graph of the fixed-capacity builder (bonds = directed edges
shorter than the bond cutoff, triplets = ordered pairs of distinct bonds at a centre), the
Fourier angle basis (triton_threebody_fourier.py), the triplet gather and the segment sums
angles -> bonds -> atoms.

Model (per layer t; atom features h [N, C], bond features eps [E, C] on every directed edge):
  edge e = (centre i <- neighbour j): vec, r, u = vec / r, ef_n = sqrt(2/rc) sin(n pi r/rc)/r fc(r)
  (n = 1..8), fc the polynomial cutoff 1 - 21x^5 + 35x^6 - 15x^7 at rc = 6 A; bond envelope
  s(r) = the same polynomial at rb (bonds: r < rb), 0 on other rows.
  triplet k = (i; bond b1, bond b2): alpha_k = [1/sqrt2, sin(theta f), cos(theta f)] / sqrt(pi),
  theta = acos((u_b1 . u_b2)(1 - 1e-6)), f = 1..F
  h = embedding[Z]; eps = ef We
  three-body:  z3_k = eps_b1 W3a + eps_b2 W3b + h_i W3c + alpha_k W3d        ([T, C])
               eps_b += (1 / avg_angles) sum_{k: b1 = b} silu(z3_k) s_b1 s_b2    (angles -> bonds)
  atom update: z2_e = h_j W2a + h_i W2b + eps_e W2c                           ([E, C])
               h_i += (1 / avg_neighbors) sum_{e: centre i} silu(z2_e) fc_e         (edges -> atoms)
  readout:     E_i = e0[Z_i] + h_i . wr
Random init from ``torch.Generator().manual_seed(seed)``.

Evaluation. Both pre-activations are sums of products of one feature row with one weight block, so
the products are formed where the feature lives and gathered, never on the edge or triplet rows:
z3_k = U[b1] + V[b2] + H[i] + aw_k with U = eps W3a, V = eps W3b on the bond rows and H = h W3c per
atom; z2_e = P[j] + Q[i] + (eps_e W2c) with P = h W2a, Q = h W2b per atom. eps_e differs from ef_e We
on the bond rows only (about a tenth of the edges): on the others the last term is ef_e (We W2c), an
n_basis-term sum in the edge kernel, and eps exists on the bond rows alone.

dE/dpos is formed by explicit VJP kernels (one autograd node). Atom update: gz2 per edge, its
per-centre and per-sender sums, the cutoff's gradient and, on the rows that are no bonds, the basis
gradient gz2 (We W2c)^T. Three-body update: per triplet gz3 and the envelope terms, per bond its sums
over the triplets as first and as second bond (gU, gV), per atom its sum. Then one product per layer
on the bond rows, geps += [gz2 | gU' | gV'] [W2c; W3a'; W3b']^T (' = the next layer's), and one on the
atoms, gh += [S_src | S_dst | S_tri] [W2a; W2b; W3c]^T. The Fourier VJP runs once over all layers'
angle gradients.
"""
from __future__ import annotations

import math
from dataclasses import dataclass, field

import torch
from torch import Tensor, nn
from torch.autograd import Function

from fastmd_amd import _abi
from fastmd_amd.adapters.protocol import (CapacityStep, CaptureContract, GraphBatch, PaddingRule, TopologySpec,
                                         require_atom_rows, system_rows)
from fastmd_amd.ops.csr_segment_sum import Csr, _prep_off, _prep_perm
from fastmd_amd.ops.threebody import LineGraph, fourier_line_vjp
from fastmd_amd.ops.wide_gemm import gemm, gemm_group, split_planes

_ELEMENTS = 118
# pairs and triplets in tiers of 128 with at least 128 of padding, held at 1.01x the pair and 1.06x
# the triplet demand (the CHGNet adapter's tiers, fastmd/models/chgnet.py:25-30)
_CAPACITY_STEP = CapacityStep(u_step=128, min_pad_u=128, u_thermal_factor=1.01, t_step=128, min_pad_t=128,
                              t_thermal_factor=1.06)


@dataclass(frozen=True)
class ThreeBodyConfig:
    channels: int = 64
    num_interactions: int = 4
    n_basis: int = 8
    cutoff: float = 6.0
    bond_cutoff: float = 3.0
    n_freq: int = 4  # 1 + 2 * 4 = 9 angle columns: the constant and 8 Fourier terms
    avg_num_neighbors: float = 15.0
    avg_num_angles: float = 4.0
    elements: tuple = (55, 50, 53)
    seed: int = 0


class ThreeBodyLike(nn.Module):
    """Parameters (frozen, float32), matrices stored [in, out]."""

    def __init__(self, config: ThreeBodyConfig = ThreeBodyConfig()) -> None:
        super().__init__()
        self.config = config
        C, nb, A = config.channels, config.n_basis, 1 + 2 * config.n_freq
        if C % 64 or not 64 <= C <= 256:
            raise ValueError("channels must be 64, 128, 192 or 256")
        if not 0.0 < config.bond_cutoff <= config.cutoff:
            raise ValueError("the bond cutoff must lie in (0, cutoff]")
        nel = len(config.elements)
        gen = torch.Generator().manual_seed(config.seed)

        def rnd(*shape, fan_in=None):
            std = 1.0 / math.sqrt(fan_in) if fan_in else 1.0
            return nn.Parameter(torch.randn(*shape, generator=gen) * std, requires_grad=False)

        self.embedding = rnd(nel, C)
        self.We = rnd(nb, C, fan_in=nb)
        self.layers = nn.ModuleList()
        for _ in range(config.num_interactions):
            layer = nn.Module()
            layer.W3 = rnd(3 * C + A, C, fan_in=3 * C + A)  # [eps_b1; eps_b2; h_i; alpha]
            layer.W2 = rnd(3 * C, C, fan_in=3 * C)  # [h_j; h_i; eps_e]
            self.layers.append(layer)
        self.wr = rnd(C, fan_in=C)
        self.e0 = nn.Parameter(-1.0 - torch.rand(nel, generator=gen), requires_grad=False)
        self.register_buffer("freqs", torch.arange(1, config.n_freq + 1, dtype=torch.float32))
        table = torch.full((_ELEMENTS + 1,), -1, dtype=torch.int32)
        for k, z in enumerate(config.elements):
            table[z] = k
        self.register_buffer("z_table", table)

    @property
    def fourier_scale(self) -> float:
        return math.sqrt(math.pi)

    def _cached(self, key, build):
        """Derived weight layouts, rebuilt when a parameter changes in place (version counter)."""
        params = [p for p in self.parameters()]
        stamp = tuple((p.data_ptr(), p._version) for p in params)
        cache = self.__dict__.setdefault("_layout_cache", {})
        hit = cache.get(key)
        if hit is None or hit[0] != stamp:
            hit = (stamp, build())
            cache[key] = hit
        return hit[1]

    def layouts(self) -> dict:
        C = self.config.channels

        def build():
            W3 = [layer.W3.detach() for layer in self.layers]
            W2 = [layer.W2.detach() for layer in self.layers]
            We = self.We.detach().double()
            last = len(W3) - 1
            out = {"node": [], "bond": [], "node_vjp": [], "bond_vjp": [], "rt": []}
            for t in range(last + 1):
                w3a, w3b, w3c = W3[t][:C], W3[t][C:2 * C], W3[t][2 * C:3 * C]
                w2a, w2b, w2c = W2[t][:C], W2[t][C:2 * C], W2[t][2 * C:]
                following = [] if t == last else [W3[t + 1][:C], W3[t + 1][C:2 * C]]
                # (N, K) layouts. Forward: h [W3c | W2a | W2b], eps [W2c | W3a' | W3b']
                out["node"].append(torch.cat([w3c, w2a, w2b], 1).t().contiguous())
                out["bond"].append(torch.cat([w2c, *following], 1).t().contiguous())
                # VJP: [S_src | S_dst | S_tri] [W2a; W2b; W3c]^T, [gz2 | gU' | gV'] [W2c; W3a'; W3b']^T
                out["node_vjp"].append(torch.cat([w2a, w2b, w3c], 1).contiguous())
                out["bond_vjp"].append(torch.cat([w2c, *following], 1).contiguous())
                out["rt"].append((We @ w2c.double()).float().contiguous())  # [nb, C]
            first = W3[0][:2 * C].double()
            # ef [We | We W3a | We W3b]: the bond rows' first eps, U and V; [gU | gV] [W3a; W3b]^T at the end
            out["init"] = torch.cat([We, We @ first[:C], We @ first[C:]], 1).float().contiguous()  # [nb, 3C]
            out["init_vjp"] = torch.cat([W3[0][:C], W3[0][C:2 * C]], 1).contiguous()  # [C, 2C]
            out["w3d"] = torch.cat([w[3 * C:] for w in W3], 1).contiguous()  # [A, L C]
            # the node products' weights as bf16 planes (their split-plane form)
            out["node_planes"] = [split_planes(w) for w in out["node"]]
            out["node_vjp_planes"] = [split_planes(w) for w in out["node_vjp"]]
            return out

        return self._cached("layouts", build)


@dataclass
class ThreeBodyInput:
    batch: GraphBatch
    line: LineGraph
    elem: Tensor  # int32 [rows]
    csr_src: Csr = field(default=None)  # the rows that an atom sends


def _call(name, *args):
    _abi.call(name, *args, _abi.stream_handle())


def _empty(*shape, device, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device=device)


class _Saved:
    """What the forward keeps for the VJP (the autograd ctx, or this holder outside autograd)."""


def _forward(ctx, positions: Tensor, cell: Tensor, model: ThreeBodyLike, inputs: ThreeBodyInput) -> Tensor:
    cfg = model.config
    batch, lg = inputs.batch, inputs.line
    dev = positions.device
    C, nb, L = cfg.channels, cfg.n_basis, cfg.num_interactions
    A = 1 + 2 * cfg.n_freq
    n = positions.shape[0]
    e_cap, t_cap = batch.edge_index.shape[0], lg.t_cap
    if positions.dtype != torch.float32:
        raise ValueError("the three-body model runs in float32")
    if lg.e_cap != e_cap or lg.edge_triplet_offsets is None:
        raise ValueError("the line graph does not match the edge list")
    positions = positions.detach().contiguous()
    cell = cell.detach().to(torch.float32).contiguous()
    ei, off, n_edges = batch.edge_index, batch.edge_offsets, batch.n_edges
    lay = model.layouts()
    geo = _empty(e_cap, 8, device=dev)
    ef = _empty(e_cap, nb, device=dev)
    de = _empty(e_cap, nb, device=dev)
    _call("fmd_edge_geometry_f32", positions.data_ptr(), cell.data_ptr(), system_rows(batch), ei.data_ptr(),
          batch.edge_image.data_ptr(),
          n_edges.data_ptr(), e_cap, float(cfg.cutoff), nb, geo.data_ptr(), ef.data_ptr(), de.data_ptr())
    _call("fmd_tb_bond_envelope_f32", geo.data_ptr(), lg.short_flags.data_ptr(), n_edges.data_ptr(), e_cap,
          float(cfg.bond_cutoff))
    # the angle basis of every triplet row and its products with all layers' angle blocks
    alpha = _empty(t_cap, A, device=dev)
    _call("fmd_threebody_fourier_line_f32", geo.data_ptr(), 8, lg.pair_offsets.data_ptr(), lg.short_counts.data_ptr(),
          lg.short_edge_matrix.data_ptr(), lg.bmax, lg.line_graph.data_ptr(), _abi.ptr(lg.overflow), lg.n_atoms,
          t_cap, model.freqs.data_ptr(), cfg.n_freq, model.fourier_scale, alpha.data_ptr())
    aw = gemm(alpha, lay["w3d"], b_layout=1)  # [T, L C]
    h = _empty(n, C, device=dev)
    _call("fmd_embed_f32", inputs.elem.data_ptr(), model.embedding.data_ptr(), n, C, h.data_ptr())
    inv_ang, inv_avg = 1.0 / cfg.avg_num_angles, 1.0 / cfg.avg_num_neighbors
    lines = lg.short_offsets.data_ptr(), lg.bond_rows.data_ptr()
    # per bond row [eps | eps W2c | U | V] (the other rows are never touched), per atom [H | P | Q]
    x = _empty(e_cap, 4 * C, device=dev)
    x_eps, x_c, x_u, x_v = (x[:, k * C:].data_ptr() for k in range(4))
    hpq = _empty(n, 3 * C, device=dev)
    _call("fmd_tb_bond_init_f32", ef.data_ptr(), nb, lay["init"].data_ptr(), C, *lines,
          _abi.ptr(lg.overflow), lg.n_atoms, e_cap, x_eps, 4 * C)
    saved = []
    for t in range(L):
        gemm_group([{"a": h, "b": lay["node"][t], "b_planes": lay["node_planes"][t], "out": hpq}], b_layout=0)
        z3 = _empty(t_cap, C, device=dev)
        _call("fmd_tb_bond_update_f32", x_u, x_v, 4 * C, hpq.data_ptr(), 3 * C, aw[:, t * C:].data_ptr(), L * C, C,
              geo.data_ptr(), *lines, lg.edge_triplet_offsets.data_ptr(), lg.line_graph.data_ptr(), lg.n_atoms, t_cap,
              inv_ang, z3.data_ptr(), C, x_eps, 4 * C)
        bond = lay["bond"][t]
        _call("fmd_tb_bond_product_f32", x_eps, 4 * C, C, None, 0, C, bond.data_ptr(), C, bond.shape[0], *lines,
              _abi.ptr(lg.overflow), lg.n_atoms, e_cap, x_c, 4 * C, 0)
        z2 = _empty(e_cap, C, device=dev)
        _call("fmd_tb_edge_sum_f32", hpq[:, C:].data_ptr(), 3 * C, ei.data_ptr(), ef.data_ptr(), nb,
              lay["rt"][t].data_ptr(), C, geo.data_ptr(), lg.short_flags.data_ptr(), x_c, 4 * C, off.data_ptr(), n,
              e_cap, inv_avg, z2.data_ptr(), h.data_ptr(), C)
        saved.append((z3, z2))
    energy = _empty(n, device=dev)
    _call("fmd_tb_readout_f32", h.data_ptr(), C, C, model.wr.data_ptr(), inputs.elem.data_ptr(), model.e0.data_ptr(),
          n, energy.data_ptr())
    ctx.model, ctx.inputs, ctx.saved = model, inputs, saved
    ctx.geo, ctx.de = geo, de
    ctx.n, ctx.e_cap = n, e_cap
    return energy


def _vjp(ctx, gE: Tensor | None, sign: float, stress_cell: Tensor | None = None):
    """sign * dE/dpos [n, 3] (gE None: the gradient of the plain sum of the node energies); with
    ``stress_cell`` (the unstrained float32 cell) also the stress [3, 3]: ``(forces, stress)``."""
    model, inputs = ctx.model, ctx.inputs
    cfg = model.config
    lg, batch = inputs.line, inputs.batch
    C, nb, L = cfg.channels, cfg.n_basis, cfg.num_interactions
    n, e_cap, t_cap = ctx.n, ctx.e_cap, lg.t_cap
    dev = ctx.geo.device
    geo = ctx.geo
    lay = model.layouts()
    inv_ang, inv_avg = 1.0 / cfg.avg_num_angles, 1.0 / cfg.avg_num_neighbors
    off = batch.edge_offsets

    gh = _empty(n, C, device=dev)
    _call("fmd_tb_readout_bwd_f32", _abi.ptr(gE), 1.0, model.wr.data_ptr(), C, n, gh.data_ptr(), C)
    # bond rows only; stored by the first layer the loop takes (the last), added to by the others
    geps = _empty(e_cap, C, device=dev)
    guv = _empty(e_cap, 2 * C, device=dev)  # [gU | gV], bond rows only
    gef = _empty(e_cap, nb, device=dev)
    gfc = _empty(e_cap, device=dev)
    gs = _empty(e_cap, device=dev)  # written on the bond rows only (read there only)
    gz3_all = _empty(t_cap, L * C, device=dev)
    gz2 = _empty(e_cap, C, device=dev)
    sums = _empty(n, 3 * C, device=dev)  # [S_src | S_dst | S_tri]
    gsw = _empty(t_cap, 2, device=dev)
    lines = lg.short_offsets.data_ptr(), lg.bond_rows.data_ptr()
    sent, sent_off = _prep_perm(inputs.csr_src.perm), _prep_off(inputs.csr_src.off)

    def bond_product(a0, k0, a1, weight, accumulate):
        _call("fmd_tb_bond_product_f32", a0.data_ptr(), k0, k0, _abi.ptr(a1), 2 * C, weight.shape[1],
              weight.data_ptr(), weight.shape[1], C, *lines, _abi.ptr(lg.overflow), n, e_cap, geps.data_ptr(), C,
              accumulate)

    for t in reversed(range(L)):
        z3, z2 = ctx.saved[t]
        later = 0 if t == L - 1 else 1
        _call("fmd_tb_edge_sum_bwd_f32", gh.data_ptr(), C, z2.data_ptr(), nb, lay["rt"][t].data_ptr(), C,
              geo.data_ptr(), off.data_ptr(), n, e_cap, inv_avg, gz2.data_ptr(), sums[:, C:].data_ptr(), 3 * C,
              gfc.data_ptr(), gef.data_ptr(), later)
        bond_product(gz2, C, guv if later else None, lay["bond_vjp"][t], later)
        # gz3 per triplet (this layer's column block) and its envelope terms
        gz3 = gz3_all[:, t * C:(t + 1) * C]
        _call("fmd_tb_triplet_bwd_f32", geps.data_ptr(), C, z3.data_ptr(), C, C, geo.data_ptr(),
              lg.line_graph.data_ptr(), lg.pair_offsets.data_ptr(), n, t_cap, inv_ang, gz3.data_ptr(), L * C,
              gsw.data_ptr())
        # per bond gU, gV and the envelope terms, per atom the sent edges' gz2 and the triplets' gz3
        _call("fmd_tb_vjp_sums_f32", gz3.data_ptr(), L * C, C, gsw.data_ptr(), *lines,
              lg.edge_triplet_offsets.data_ptr(), lg.second_perm.data_ptr(), lg.pair_offsets.data_ptr(), n, t_cap,
              guv.data_ptr(), 2 * C, gs.data_ptr(), later, gz2.data_ptr(), sent_off.data_ptr(),
              sent.data_ptr(), e_cap, sums.data_ptr(), sums[:, 2 * C:].data_ptr(), 3 * C)
        gemm_group([{"a": sums, "b": lay["node_vjp"][t], "b_planes": lay["node_vjp_planes"][t], "out": gh,
                     "accumulate": True}], b_layout=0)
    bond_product(guv, 2 * C, None, lay["init_vjp"], 1)
    _call("fmd_tb_bond_basis_f32", geps.data_ptr(), C, C, model.We.data_ptr(), nb, *lines, n, e_cap, gef.data_ptr())
    # the angle basis: all layers' angle gradients at once, then the Fourier VJP (short rows)
    galpha = gemm(gz3_all, lay["w3d"], b_layout=0)  # [T, A]
    gu = _empty(e_cap, 3, device=dev)  # written on the bond rows only (read there only)
    fourier_line_vjp(galpha, geo[:, :3], lg, model.freqs, model.fourier_scale, out=gu, accumulate=False)
    gvec = None if stress_cell is None else _empty(e_cap, 3, device=dev)  # the virial reads it
    forces = _empty(n, 3, device=dev)
    _call("fmd_tb_edge_forces_f32", geo.data_ptr(), ctx.de.data_ptr(), nb, gef.data_ptr(), nb, gu.data_ptr(), 3,
          gfc.data_ptr(), gs.data_ptr(), lg.short_flags.data_ptr(), sent_off.data_ptr(), sent.data_ptr(),
          batch.n_edges.data_ptr(), e_cap, n, sign, forces.data_ptr(), _abi.ptr(gvec))
    if stress_cell is None:
        return forces
    from fastmd_amd.engine.energy_derivative import edge_stress

    # the angles enter through the bond unit vectors, whose gradient is part of gvec: the virial
    # of the edge vectors is the whole strain derivative
    return forces, edge_stress(geo, gvec, batch.n_edges, stress_cell)


class _ThreeBodyEnergy(Function):
    """positions -> node energies [rows]; backward: dE/dpos by the VJP kernels."""

    @staticmethod
    def forward(ctx, positions, cell, model: ThreeBodyLike, inputs: ThreeBodyInput):
        return _forward(ctx, positions, cell, model, inputs)

    @staticmethod
    def backward(ctx, gE):
        gE = gE.detach().to(torch.float32).contiguous()
        return _vjp(ctx, gE, 1.0), None, None, None


class ThreeBodyAdapter:
    """The three-body model as a ModelAdapter with an EnergyTap (chgnet.py's surface: line-graph
    topology, far self-loop padding, pair and triplet capacity tiers)."""

    name = "threebody_like"
    compiled = False

    def __init__(self, module: ThreeBodyLike | None = None, *, config: ThreeBodyConfig | None = None,
                 device: torch.device | str = "cuda") -> None:
        module = module if module is not None else ThreeBodyLike(config or ThreeBodyConfig())
        self.module = module.to(device).eval()
        for p in self.module.parameters():
            p.requires_grad_(False)

    def topology_spec(self) -> TopologySpec:
        cfg = self.module.config
        return TopologySpec(cutoff=float(cfg.cutoff), num_interactions=int(cfg.num_interactions),
                            triplet_cutoff=float(cfg.bond_cutoff), undirected_pairs=True, model_dtype="float32",
                            edge_order="sorted")

    def padding_rule(self) -> PaddingRule:
        return PaddingRule("far_self_loops")

    def capacity_step(self) -> CapacityStep:
        return _CAPACITY_STEP

    def capture_contract(self) -> CaptureContract:
        return CaptureContract(sync_free=True, exact_cutoff=True, accuracy_class="fp32_noise",
                               force_mode="engine_autograd", stress_unit="eV/A^3", compiled="none")

    def isolated_atom_policy(self) -> str:
        return "model"

    def reference_energies(self) -> Tensor:
        row = torch.full((1, _ELEMENTS), float("nan"), dtype=torch.float64)
        for k, z in enumerate(self.module.config.elements):
            row[0, z - 1] = float(self.module.e0[k])
        return row

    def prepare(self, batch: GraphBatch) -> ThreeBodyInput:
        """Aliases of the batch and its line graph, the element index of every row (host check of
        the species, outside any graph) and the CSR of the rows by sender."""
        if batch.positions is None or batch.edge_offsets is None or batch.edge_reverse is None:
            raise ValueError("the three-body model needs a fixed-capacity batch with its CSR")
        require_atom_rows(batch, "three-body")
        if batch.line is None or batch.line.edge_triplet_offsets is None:
            raise ValueError("the three-body model reads a line graph (a builder with line_graph_cutoff)")
        if abs(float(batch.triplet_cutoff) - float(self.module.config.bond_cutoff)) > 1e-12:
            raise ValueError(f"line graph cutoff {batch.triplet_cutoff} != the model's bond cutoff "
                             f"{self.module.config.bond_cutoff}")
        species = batch.species.long()
        table = self.module.z_table.to(species.device)
        if bool(((species < 1) | (species > _ELEMENTS)).any()) or bool((table[species.clamp(1, _ELEMENTS)] < 0).any()):
            raise ValueError(f"the three-body model supports atomic numbers {list(self.module.config.elements)}")
        elem = table[species].to(torch.int32).contiguous()
        rows = batch.edge_index.shape[0]
        return ThreeBodyInput(batch=batch, line=batch.line, elem=elem,
                              csr_src=Csr(batch.edge_offsets, batch.edge_reverse, rows))

    def node_energy(self, inputs: ThreeBodyInput, positions: Tensor, cell: Tensor) -> Tensor:
        if cell.requires_grad:
            raise NotImplementedError("stress (a strained cell) is not supported by the three-body kernels")
        return _ThreeBodyEnergy.apply(positions, cell, self.module, inputs)

    def energy_and_forces(self, inputs: ThreeBodyInput, positions: Tensor, cell: Tensor,
                          segments=1) -> tuple[Tensor, Tensor]:
        """(E [1] float64, F = -dE/dpos [rows, 3]) by the forward and VJP kernels, without autograd."""
        from fastmd_amd.engine.energy_derivative import sum_f64_segments

        saved = _Saved()
        energies = _forward(saved, positions.detach(), cell.detach(), self.module, inputs)
        energy = sum_f64_segments(energies, segments)  # one energy per replica or system
        return energy, _vjp(saved, None, -1.0)

    def energy_forces_stress(self, inputs: ThreeBodyInput, positions: Tensor, cell: Tensor):
        """``energy_and_forces`` plus the stress dE/d(strain) / V [3, 3] float32 of one system
        (energy_derivative.py:110-140)."""
        from fastmd_amd.engine.energy_derivative import sum_f64_into

        saved = _Saved()
        energies = _forward(saved, positions.detach(), cell.detach(), self.module, inputs)
        energy = sum_f64_into(energies)
        forces, stress = _vjp(saved, None, -1.0, stress_cell=cell.detach().to(torch.float32).contiguous())
        return energy, forces, stress
