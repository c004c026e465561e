"""MACE-ICTC baseline model (bridge-U product) on the MI355X kernels.

Composition follows the reference's ``PureCartesianICTDFix`` for the route
``create_model`` builds (mace_ictc/hp/runtime.py:6-83 ->
models/factory.py:8-160 -> models/mace/backbone.py:60-726, forward :860-1250):

  h0 = embedding[species]                                            (backbone.py:1016-1020)
  per interaction i (layers.py:1042-1368):
    x  = linear_up(h)                       per-degree C x C
    m  = scatter_dst( TP(x[src], Y(e), fc(radial(r))) * mask )     CSR message kernel
    m  = message_linear(m) / avg_num_neighbors                      path-preserving linear
    sc = self_connection[species](h_l0)                             element-conditioned, l = 0
  product i (products.py:792-841): h = linear(SC(m)) + sc on l = 0   (common.py:82-106)
  readout: layer < last: Linear(C,1) on l = 0 (pure_cartesian_ictd_layers.py:89-115);
           last: Linear(C,16) -> SiLU*1.679 -> Linear(16,1)          (heads.py:12-27)
  atomic energy = sum of layer readouts.

Parameter names, shapes and initialisation match the reference so state
dicts line up.  Node features use the packed component-major layout of the
kernels ([N, sum_l (2l+1) * C], component l*l+m at columns (l*l+m)*C..).
"""
from __future__ import annotations

import math
import weakref
from typing import Dict, List

import torch
import torch.nn as nn
import torch.nn.functional as F

from ictc_o3.basis import tables
from ictc_o3.basis.ictd_irreps import EdgeWeightedPathPreservingTensorProduct
from ictc_o3.ops import tensor_product as tpo
from ictc_o3.ops.harmonics import harmonics_packed
from ictc_o3.ops.linear import species_rows, take_scalars
from ictc_o3.ops.radial_mlp import EdgeLengths, edge_linear, hidden_supported, radial_mlp_lengths
from ictc_o3.ops.symmetric_contraction import ICTDBridgeUSymmetricContractionSO3

SILU_SCALE = 1.6791767923989418   # _Normalize2MomSiLU (layers.py:307-314)


class NormalizedSiLU(nn.Module):
    _scale = SILU_SCALE

    def forward(self, x):
        from ictc_o3.ops.activation import normalized_silu
        return normalized_silu(x, self._scale)


def _mace_linear_init(linear: nn.Linear):
    """common.py:_init_mace_style_linear_: N(0, 1/sqrt(fan_in))."""
    with torch.no_grad():
        nn.init.normal_(linear.weight, mean=0.0, std=1.0 / math.sqrt(float(linear.in_features)))


def degree_linear(x, weights: List[torch.Tensor], C: int, lmax: int, scale: float = 1.0, first_order=False):
    """Per-degree channel map on the packed layout: out[n, l*l+m, :] = scale * W_l @ x[n, l*l+m, :].

    first_order=True runs the MFMA kernel with a first-derivative adjoint; otherwise the same kernel with
    adjoints differentiable to any order (the composable per-degree form where the kernel does not apply)."""
    from ictc_o3.ops.linear import degree_linear_any, degree_linear_fast
    return (degree_linear_fast if first_order else degree_linear_any)(x, weights, C, lmax, scale)


class ChannelLinear(nn.Module):
    """EquivariantChannelLinearSO3 (ictd_irreps.py:207-227): adapters[str(l)] = Linear(C, C)."""

    def __init__(self, channels, lmax):
        super().__init__()
        self.channels, self.lmax = channels, lmax
        self.adapters = nn.ModuleDict({str(l): nn.Linear(channels, channels, bias=False) for l in range(lmax + 1)})
        with torch.no_grad():
            for a in self.adapters.values():
                nn.init.eye_(a.weight)       # interaction_init="identity" (common.py:71-114)

    def forward(self, x, first_order=False):
        return degree_linear(x, [self.adapters[str(l)].weight for l in range(self.lmax + 1)], self.channels,
                             self.lmax, first_order=first_order)


class PathPreservingLinear(nn.Module):
    """PathPreservingLinearSO3 (layers.py:317-355): weights[str(l)] [C, count_l*C]."""

    def __init__(self, counts: Dict[int, int], channels: int, lmax: int):
        super().__init__()
        self.counts, self.channels, self.lmax = counts, channels, lmax
        self.weights = nn.ParameterDict()
        for l in range(lmax + 1):
            k = counts.get(l, 0) * channels
            w = nn.Parameter(torch.empty(channels, k))
            if k:
                nn.init.normal_(w, mean=0.0, std=1.0 / math.sqrt(float(k)))
            self.weights[str(l)] = w

    def forward(self, m, scale: float, first_order=False):
        from ictc_o3.ops.linear import path_linear_any, path_linear_fast
        return (path_linear_fast if first_order else path_linear_any)(
            m, [self.weights[str(l)] for l in range(self.lmax + 1)], self.counts, self.channels, self.lmax, scale)


class ElementConditionedLinear(nn.Module):
    """ElementConditionedLinearSO3 (layers.py:21-87), identity init (common.py:128-142)."""

    def __init__(self, num_elements, channels, lmax):
        super().__init__()
        self.num_elements, self.channels, self.lmax = num_elements, channels, lmax
        self.weights = nn.ParameterDict({str(l): nn.Parameter(
            torch.eye(channels).unsqueeze(0).repeat(num_elements, 1, 1)) for l in range(lmax + 1)})
        self.bias = None

    def forward_l0(self, x0, species):
        """out[n, o] = sum_i W[s_n, o, i] x0[n, i] for the scalar block."""
        from ictc_o3.ops.linear import species_linear
        return species_linear(x0, self.weights["0"], species)


class ProductLinear(nn.Module):
    """e3nn o3.Linear on Cx0e + Cx1o + ... : flat weight, per-degree [C_in, C_out] blocks, 1/sqrt(C) scale."""

    def __init__(self, channels, lmax):
        super().__init__()
        self.channels, self.lmax = channels, lmax
        self.weight = nn.Parameter(torch.randn((lmax + 1) * channels * channels))

    def blocks(self):
        C = self.channels
        return [self.weight[l * C * C:(l + 1) * C * C].view(C, C).t() for l in range(self.lmax + 1)]

    def forward(self, x, first_order=False):
        return degree_linear(x, self.blocks(), self.channels, self.lmax, 1.0 / math.sqrt(self.channels),
                             first_order=first_order)


class Interaction(nn.Module):
    def __init__(self, *, channels, edge_lmax, input_lmax, sc_lmax, number_of_basis, num_elements,
                 radial_hidden=(64, 64, 64), avg_num_neighbors=50.0):
        super().__init__()
        self.channels, self.lmax, self.input_lmax = channels, edge_lmax, input_lmax
        self.target_lmax, self.sc_lmax = edge_lmax, sc_lmax
        self.avg_num_neighbors = avg_num_neighbors
        self.linear_up = ChannelLinear(channels, input_lmax)
        paths = tables.natural_paths(input_lmax, edge_lmax, edge_lmax)
        self.tp = EdgeWeightedPathPreservingTensorProduct(channels=channels, lmax=edge_lmax, allowed_paths=paths,
                                                          internal_compute_dtype=torch.float32)
        with torch.no_grad():
            self.tp.weight.fill_(1.0)
        self.tp.weight.requires_grad_(False)     # freeze_conv_tp_weight=True (runtime.py:76)
        sizes = (number_of_basis, *radial_hidden, self.tp.num_paths * channels)
        layers = []
        for k, (a, b) in enumerate(zip(sizes, sizes[1:])):
            layers.append(nn.Linear(a, b, bias=False))
            if k < len(sizes) - 2:
                layers.append(NormalizedSiLU())
        self.fc = nn.Sequential(*layers)
        for m in self.fc:
            if isinstance(m, nn.Linear):
                _mace_linear_init(m)
        self.message_linear = PathPreservingLinear(dict(self.tp.path_counts_by_l), channels, edge_lmax)
        self.self_connection = ElementConditionedLinear(num_elements, channels, sc_lmax)
        self._spec = None

    def spec(self):
        if self._spec is None:
            self._spec = tpo.make_spec(self.input_lmax, self.lmax, self.lmax, self.channels, None)
        return self._spec

    def entry(self, h):
        """(linear_up(h), h[:, :C]) from one first-order op whose adjoint merges both gradients, or None
        where the input has only scalar columns or the MFMA linear does not apply."""
        from ictc_o3.ops.linear import layer_entry_fast
        a = self.linear_up
        return layer_entry_fast(h, [a.adapters[str(l)].weight for l in range(a.lmax + 1)], self.channels, a.lmax)

    def forward(self, h, species, Y, radial, topo, mask, r=None, radial_cfg=None, forces_only=False,
                basis_scale=1.0, entry=None, species_table=None):
        """radial: [E, K] basis (composable path) or None with r / radial_cfg (fused first-order path;
        basis_scale multiplies the radial basis there).  entry: (linear_up(h), h[:, :C]) from entry().
        species_table: [S, C] with linear_up(h)[n] == species_table[species[n]] (the first layer, whose
        input is the species embedding), which lets the message run in its species form."""
        C = self.channels
        first_order = radial is None
        if entry is not None and entry[0] is not None:
            x, h0 = entry
        else:
            from ictc_o3.ops.linear import take_scalars
            x = self.linear_up(h, first_order)
            h0 = entry[1] if entry is not None else take_scalars(h, C)
        if radial is None and forces_only:
            m = tpo.radial_message(x, Y, r, self.fc, self.spec(), topo, mask, radial_cfg, basis_scale,
                                   species=None if species_table is None else (species_table, species))
        else:
            if radial is None:
                from ictc_o3.ops.radial_mlp import radial_gates
                gates = radial_gates(r, self.fc, *radial_cfg, basis_scale=basis_scale)
            elif isinstance(radial, EdgeLengths):
                gates = radial_mlp_lengths(r, self.fc, *radial_cfg, basis_scale=basis_scale)
            else:
                from ictc_o3.ops.radial_mlp import radial_mlp
                gates = radial_mlp(radial, self.fc)
            m = tpo.message(x, Y, gates, self.spec(), topo, mask)
        message = self.message_linear(m, 1.0 / max(self.avg_num_neighbors, 1e-8), first_order)
        sc = self.self_connection.forward_l0(h0, species)
        return message, sc


class Product(nn.Module):
    def __init__(self, *, num_elements, channels, lmax, target_lmax, correlation):
        super().__init__()
        self.channels, self.target_lmax = channels, target_lmax
        self.symmetric_contractions = ICTDBridgeUSymmetricContractionSO3(
            num_elements=num_elements, channels=channels, lmax=lmax, target_lmax=target_lmax,
            correlation=correlation)
        self.linear = ProductLinear(channels, target_lmax)

    def forward(self, message, sc, species, first_order=False):
        out = self.linear(self.symmetric_contractions.contract(message, species, shared_order=True), first_order)
        C = self.channels
        if out.shape[1] == C:
            return out + sc
        # in place on the linear's fresh output (no backward saves it): no concatenation copy
        if first_order:
            from ictc_o3.ops.linear import add_scalars_
            return add_scalars_(out, sc)
        from ictc_o3.ops.linear import add_scalars_any_
        return add_scalars_any_(out, sc)


class ScalarReadout(nn.Module):
    """EquivariantScalarReadoutSO3: readout = Linear(C, 1) on the l=0 block."""

    def __init__(self, channels):
        super().__init__()
        self.readout = nn.Linear(channels, 1, bias=False)
        nn.init.normal_(self.readout.weight, mean=0.0, std=1.0 / math.sqrt(channels))

    def forward(self, h0):
        return edge_linear(h0, self.readout.weight)


class MACEStyleReadout(nn.Module):
    """MACEStyleScalarReadoutSO3: Linear(C,16) -> SiLU*1.679 -> Linear(16,1)."""

    def __init__(self, channels, hidden=16):
        super().__init__()
        self.linear_1 = nn.Linear(channels, hidden, bias=False)
        self.activation = NormalizedSiLU()
        self.linear_2 = nn.Linear(hidden, 1, bias=False)
        _mace_linear_init(self.linear_1)
        _mace_linear_init(self.linear_2)

    def forward(self, h0):
        return edge_linear(self.activation(edge_linear(h0, self.linear_1.weight)), self.linear_2.weight)


def shift_vectors(shifts: torch.Tensor, cell: torch.Tensor, batch: torch.Tensor, edge_src: torch.Tensor):
    """Cartesian image shifts [E, 3] = shifts [E, 3] (lattice coordinates) . cell of the edge's graph.

    Topology.pair_edges lets an edge and its reverse (shift -S) share one row of
    radial gates, which is only exact when their lengths are bitwise equal.  They
    are because this form is odd in the shift bit for bit: each component is a
    sum of three products s_k * c_kj in a fixed order, and negating every s_k
    negates every product and every partial sum exactly (on the device: the
    kernel ictc_shift_vectors, every operation rounded on its own).  A library GEMM or an
    FMA-contracted form need not keep that (its order or fusion may differ with
    the operand's sign pattern), so do not change it without re-running the
    shared-row bitwise tests.
    """
    # the kernel carries no gradient: a caller differentiating in the shifts or the cell (the LAMMPS core
    # passes its edge vectors as shifts) takes the torch form
    if (shifts.is_cuda and shifts.dtype == torch.float32
            and not (torch.is_grad_enabled() and (cell.requires_grad or shifts.requires_grad))):
        from ictc_o3.ops.geometry import shift_vectors as native_shift_vectors
        return native_shift_vectors(shifts, cell, batch, edge_src)
    if cell.shape[0] == 1:   # [E, 3] x [3, 3] as three broadcast products (no library GEMM)
        return (shifts.unsqueeze(-1) * cell[0].to(shifts.dtype)).sum(1)
    # per-edge cell rows without a batched 1x3x3 GEMM per edge
    return (shifts.unsqueeze(-1) * cell[batch[edge_src]].to(shifts.dtype)).sum(1)


class PureCartesianICTDFix(nn.Module):
    """The baseline MACE-ICTC backbone restricted to the create_model route."""

    def __init__(self, *, channels=64, lmax=2, edge_lmax=None, num_interactions=2, correlation=3,
                 atomic_numbers=(1, 6, 8), cutoff=5.0, avg_num_neighbors=50.0, number_of_basis=8,
                 polynomial_cutoff_p=5, readout_hidden=16, radial_sqrt_num_basis=False):
        super().__init__()
        # the historical sqrt(num_basis) radial norm (radial_basis.py:87-91); create_model leaves it off
        self.radial_sqrt_num_basis = bool(radial_sqrt_num_basis)
        self.radial_basis_scale = math.sqrt(number_of_basis) if radial_sqrt_num_basis else 1.0
        edge_lmax = lmax if edge_lmax is None else edge_lmax
        self.channels, self.lmax, self.ictd_fix_edge_lmax = channels, lmax, edge_lmax
        self.num_interaction, self.max_radius = num_interactions, float(cutoff)
        self.number_of_basis, self.polynomial_cutoff_p = number_of_basis, polynomial_cutoff_p
        self.avg_num_neighbors = float(avg_num_neighbors)
        self.atomic_numbers = tuple(sorted({int(z) for z in atomic_numbers}))
        self.num_elements = len(self.atomic_numbers)
        table = torch.full((max(119, max(self.atomic_numbers) + 1),), -1, dtype=torch.long)
        for i, z in enumerate(self.atomic_numbers):
            table[z] = i
        self.register_buffer("atomic_number_to_index", table, persistent=False)
        self.node_embedding = nn.Linear(self.num_elements, channels, bias=False)
        self.interactions = nn.ModuleList()
        self.products = nn.ModuleList()
        for i in range(num_interactions):
            target = lmax if i < num_interactions - 1 else 0
            input_lmax = 0 if i == 0 else lmax
            self.interactions.append(Interaction(
                channels=channels, edge_lmax=edge_lmax, input_lmax=input_lmax, sc_lmax=0,
                number_of_basis=number_of_basis, num_elements=self.num_elements,
                avg_num_neighbors=self.avg_num_neighbors))
            self.products.append(Product(num_elements=self.num_elements, channels=channels, lmax=edge_lmax,
                                         target_lmax=target, correlation=correlation))
        self.layer_energy_readouts = nn.ModuleList([ScalarReadout(channels) for _ in range(num_interactions - 1)])
        self.last_layer_energy_readout = MACEStyleReadout(channels, readout_hidden)

    # -- geometry ---------------------------------------------------------------
    def radial_embedding(self, r):
        """Bessel basis x MACE polynomial cutoff (radial_basis.py:11-92, sqrt_num_basis_norm=False)."""
        from ictc_o3.ops.activation import radial_embedding
        return radial_embedding(r, self.max_radius, self.number_of_basis, self.polynomial_cutoff_p)

    def species_indices(self, A):
        """Compact species [N] of the atomic numbers, validated (backbone.py:996-1009)."""
        A_long = A.long()
        # skip_input_validation drops the validation's host syncs.  The
        # same live tensor object with an unchanged version counter is validated once: MD and training
        # loops pass one atomic-number tensor every step, and a sync per step would stall the launches.
        seen = getattr(self, "_validated_z", None)
        validate = not getattr(self, "skip_input_validation", False) and not (
            seen is not None and seen[0]() is A and seen[1] == A._version)
        if validate and A_long.numel() > 0:
            top = int(A_long.max().item())
            if top >= self.atomic_number_to_index.numel():
                raise ValueError(
                    f"Encountered atomic number {top}, but compact mapping supports only up to "
                    f"{self.atomic_number_to_index.numel() - 1}. atomic_numbers={self.atomic_numbers}")
            if int(A_long.min().item()) < 0:
                bad = torch.unique(A_long[A_long < 0]).tolist()
                raise ValueError(f"Encountered atomic numbers without compact mapping: {bad}. "
                                 f"Configured atomic_numbers={self.atomic_numbers}")
        species = self.atomic_number_to_index[A_long]
        if validate:
            if bool(torch.any(species < 0)):
                bad = torch.unique(A_long[species < 0]).tolist()
                raise ValueError(f"Encountered atomic numbers without compact mapping: {bad}. "
                                 f"Configured atomic_numbers={self.atomic_numbers}")
            self._validated_z = (weakref.ref(A), A._version)
        return species

    def forward(self, pos, A, batch, edge_src, edge_dst, edge_shifts, cell, *, topology=None, second_order=True,
                forces_only=False):
        """Per-atom energies [N, 1].

        forces_only=True (with second_order=False) tells the fused path that the
        backward will ask for position gradients and no parameter gradients: the
        radial gates are then written with their derivative along r, and the
        message adjoint forms dE/dr without the gate gradient.  A backward that
        does ask for parameter gradients stays correct (it takes the ordinary
        route), only slower.

        second_order=False allows the fused radial-MLP kernel, whose adjoint
        supports first derivatives only (forces, parameter gradients); the
        default keeps every operator differentiable to second order.
        """
        N = pos.shape[0]
        species = self.species_indices(A)
        if topology is None:
            # spatial row order for one periodic system; batched graphs keep index order (their
            # atoms are contiguous per graph, and the graphs' coordinates overlap)
            topology = tpo.Topology(edge_src, edge_dst, N, positions=pos if cell.shape[0] == 1 else None)
        from ictc_o3.ops.radial_mlp import fused_supported
        fused = (not second_order and self.number_of_basis == 8
                 and all(fused_supported(inter.fc) for inter in self.interactions))
        if fused and forces_only and tpo.PAIR_GATES:
            # an edge and its reverse share one row of radial gates (equal lengths, bitwise); enqueued first,
            # so the GPU runs the pairing while the host prepares the geometry launches
            topology.pair_edges(edge_shifts)
        shift_vec = shift_vectors(edge_shifts.to(pos.dtype), cell, batch, edge_src)
        r_first = Y_first = None
        if second_order or pos.dtype != torch.float32:
            if pos.dtype == torch.float32 and pos.is_cuda:
                from ictc_o3.ops.geometry import edge_vectors
                vec = edge_vectors(pos, shift_vec, topology)
            else:
                vec = pos[edge_dst] - pos[edge_src] + shift_vec
            from ictc_o3.ops.geometry import edge_unit
            r, n = edge_unit(vec)   # r = |vec|, n = vec / max(r, 1e-8), derivatives to any order
            mask = (r <= self.max_radius).to(pos.dtype)
            Y = harmonics_packed(n, self.ictd_fix_edge_lmax)
        else:
            # first order: edge geometry and harmonics in one kernel, one per-edge adjoint; with two or more
            # layers, the first layer takes its own r and Y outputs so that the adjoint adds the two layers'
            # cotangents in its kernel
            from ictc_o3.ops.geometry import edge_harmonics
            if self.num_interaction >= 2:
                r, r_first, Y, Y_first, mask = edge_harmonics(pos, shift_vec, topology, self.max_radius,
                                                              self.ictd_fix_edge_lmax, uses=2)
            else:
                r, Y, mask = edge_harmonics(pos, shift_vec, topology, self.max_radius, self.ictd_fix_edge_lmax)
        if fused:
            radial = None
        elif (tpo.FUSED_HIDDEN and self.number_of_basis == 8
              and all(hidden_supported(inter.fc, r) for inter in self.interactions)):
            # second derivatives: the radial MLP's hidden layers on the fused kernels (lengths in, not the basis)
            radial = EdgeLengths()
        else:
            radial = self.radial_embedding(r)
        if isinstance(radial, torch.Tensor) and self.radial_basis_scale != 1.0:
            radial = radial * self.radial_basis_scale
        radial_cfg = (self.max_radius, self.polynomial_cutoff_p, SILU_SCALE)
        h = species_rows(self.node_embedding.weight.t(), species)
        energy = None
        for i, (inter, prod) in enumerate(zip(self.interactions, self.products)):
            # first-order route: the scalar columns come out of the next layer's entry op (one merged
            # adjoint instead of slice gradients), so layer i - 1's energy readout is taken here, in order
            entry = inter.entry(h) if radial is None else None
            if entry is None:   # the scalar columns taken once for the readout and the self connection
                entry = (None, take_scalars(h, self.channels))
            if i > 0:
                e = self.layer_energy_readouts[i - 1](entry[1])
                energy = e if energy is None else energy + e
            table = None
            if i == 0 and radial is None and forces_only and inter.input_lmax == 0:
                # the first layer's input is the species embedding: its linear_up rows per species
                with torch.no_grad():
                    table = inter.linear_up(self.node_embedding.weight.t().contiguous(), True)
            first = i == 0 and r_first is not None
            message, sc = inter(h, species, Y_first if first else Y, radial, topology, mask,
                                r_first if first else r, radial_cfg, forces_only,
                                self.radial_basis_scale, entry=entry, species_table=table)
            h = prod(message, sc, species, first_order=radial is None)
        e = self.last_layer_energy_readout(h if h.shape[1] == self.channels else h[:, :self.channels])
        return e if energy is None else energy + e
