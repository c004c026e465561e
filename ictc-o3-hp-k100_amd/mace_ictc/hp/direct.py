"""Energy and forces of the whole model as one forward and one adjoint sweep, without autograd.

energy_and_forces(training=False) (runtime.py) returns detached results, so nothing outside the call can see
the graph that autograd would record; for small systems recording it and running it back (a Function object,
saved tensors and a node per operation) is most of the step's host time, several times the GPU's.  Here the
same native operators run in the same order forward, and their adjoints in reverse, on plain tensors.

``energy_forces`` returns None, and the caller takes the autograd route, wherever something could observe or
change the difference: positions, cell or shifts that require gradients (their hooks), module or global
hooks, replaced or parametrised submodules, saved-tensor hooks, forward-mode, functorch and tracing contexts,
autocast, or shapes the first-order kernels do not cover.
"""
from __future__ import annotations

import torch
import torch.nn as nn
from torch.nn.modules import module as _module

from ictc_o3.ops import tensor_product as tpo
from ictc_o3.ops.activation import _silu
from ictc_o3.ops.geometry import _vector_adjoint, edge_harmonics_adjoint_raw, edge_harmonics_raw, shift_vectors
from ictc_o3.ops.linear import (_fast_ok, _species_apply, degree_layout, packed_linear_adjoint_raw,
                                packed_linear_raw, path_layout, species_order, transposed)
from ictc_o3.ops.radial_mlp import (edge_linear_adjoint_raw, edge_linear_raw, fused_supported,
                                    radial_gates_tangent)
from ictc_o3.ops.symmetric_contraction import (ICTDBridgeUSymmetricContractionSO3, MaceSymmetricContraction,
                                               _Contraction, _dx_raw, _fwd_raw, _SpeciesHolder)

DIRECT = True   # False: always the autograd route


def _plain(m, cls) -> bool:
    """m is a cls as it was built: no hooks, no forward of its own, no parametrisation (which changes the class)."""
    return (type(m) is cls and not m._forward_hooks and not m._forward_pre_hooks and not m._backward_hooks
            and not m._backward_pre_hooks and "forward" not in m.__dict__)


def _plain_model(model) -> bool:
    from mace_ictc.hp import model as M
    if not (_plain(model, M.PureCartesianICTDFix) and _plain(model.node_embedding, nn.Linear)
            and len(model.products) == len(model.interactions) == model.num_interaction
            and len(model.layer_energy_readouts) == model.num_interaction - 1):
        return False
    for inter in model.interactions:
        if not (_plain(inter, M.Interaction) and _plain(inter.linear_up, M.ChannelLinear)
                and all(_plain(a, nn.Linear) for a in inter.linear_up.adapters.values())
                and _plain(inter.fc, nn.Sequential)
                and all(_plain(m, nn.Linear if k % 2 == 0 else M.NormalizedSiLU) for k, m in enumerate(inter.fc))
                and _plain(inter.message_linear, M.PathPreservingLinear)
                and _plain(inter.self_connection, M.ElementConditionedLinear)):
            return False
    for prod in model.products:
        sc = prod.symmetric_contractions
        if not (_plain(prod, M.Product) and _plain(prod.linear, M.ProductLinear)
                and _plain(sc, ICTDBridgeUSymmetricContractionSO3)
                and _plain(sc.symmetric_contractions, MaceSymmetricContraction)
                and all(_plain(c, _Contraction) for c in sc.symmetric_contractions.contractions)
                and "contract" not in sc.__dict__):
            return False
    last = model.last_layer_energy_readout
    return (all(_plain(m, M.ScalarReadout) and _plain(m.readout, nn.Linear) for m in model.layer_energy_readouts)
            and _plain(last, M.MACEStyleReadout) and _plain(last.activation, M.NormalizedSiLU)
            and _plain(last.linear_1, nn.Linear) and _plain(last.linear_2, nn.Linear))


def _plain_context() -> bool:
    """No hooks or transforms around the call that an autograd graph would be visible to."""
    from torch.fx.experimental.proxy_tensor import get_proxy_mode
    from torch.autograd import forward_ad
    return not (_module._global_forward_hooks or _module._global_forward_pre_hooks or _module._global_backward_hooks
                or _module._global_backward_pre_hooks
                or torch._C._autograd._top_saved_tensors_default_hooks(False) is not None
                or forward_ad._current_level >= 0 or torch._C._are_functorch_transforms_active()
                or torch.compiler.is_compiling() or get_proxy_mode() is not None or torch.jit.is_tracing()
                or torch.is_anomaly_enabled() or torch.is_autocast_enabled("cuda")
                or torch._C._len_torch_dispatch_stack() or torch._C._len_torch_function_stack())


def _covered(model, pos, A, batch, edge_src, edge_dst, shifts, cell) -> bool:
    tensors = (pos, A, batch, edge_src, edge_dst, shifts, cell)
    if not (DIRECT and pos.is_cuda
            and all(type(t) is torch.Tensor and t.device == pos.device and not t.requires_grad for t in tensors)
            and pos.dtype == torch.float32 and edge_src.numel() > 0 and model.number_of_basis == 8
            and model.num_elements > 1):      # the packed linear takes no one-row species table
        return False
    C = model.channels
    for inter in model.interactions:
        counts = inter.message_linear.counts
        weights = [a.weight for a in inter.linear_up.adapters.values()] + list(inter.message_linear.weights.values())
        if not (fused_supported(inter.fc) and all(_fast_ok(pos, [w], C) for w in weights)
                and all(counts.get(l, 0) > 0 for l in range(inter.lmax + 1))):
            return False
    return all(p.dtype == torch.float32 and p.device == pos.device for p in model.parameters())


def _graph_ids(batch, graphs):
    """Starts reading the range of the graph ids; the function returned raises where one is outside [0, graphs).
    (The autograd route fails on such an id in the gather of the energies' adjoint, which these sweeps do not have.)
    Read with the call's first launches and waited for at its end, only that copy: nothing stalls for it."""
    if graphs == 1 or batch.numel() == 0 or torch.cuda.is_current_stream_capturing():
        return lambda: None      # one graph: the ids are not used; a captured stream has nothing to read yet
    host = torch.empty(2, dtype=batch.dtype, pin_memory=True)
    host.copy_(torch.stack(torch.aminmax(batch)), non_blocking=True)
    event = torch.cuda.Event()
    event.record(torch.cuda.current_stream(batch.device))

    def check():
        event.synchronize()
        low, high = host.tolist()
        if low < 0 or high >= graphs:
            raise ValueError(f"Graph ids run from {low} to {high}, outside 0..{graphs - 1}")
    return check


def _species_linear(x, weight, species):
    """ops.linear.species_linear (no autograd)."""
    S, Co, Ci = weight.shape
    if Co == Ci and Ci in (64, 128) and x.shape[0] < 2 ** 31:
        return _species_apply(x, weight, species_order(species, S), False)
    allp = edge_linear_raw(x, weight.reshape(S * Co, Ci)).reshape(x.shape[0], S, Co)
    return allp.gather(1, species.view(-1, 1, 1).expand(-1, 1, Co)).squeeze(1)


def _species_linear_adjoint(g, weight, species):
    S, Co, Ci = weight.shape
    if Co == Ci and Ci in (64, 128) and g.shape[0] < 2 ** 31:
        return _species_apply(g, weight, species_order(species, S), True)
    spread = g.new_zeros(g.shape[0], S, Co).scatter_(1, species.view(-1, 1, 1).expand(-1, 1, Co), g.unsqueeze(1))
    return edge_linear_adjoint_raw(spread.reshape(-1, S * Co), weight.reshape(S * Co, Ci))


def _c(w):
    w = w.detach()
    return w if w.is_contiguous() else w.contiguous()


class _Layer:
    """One interaction and product: forward() keeps what adjoint() reads.  The weights are read anew on each call
    (nothing tells of a write through weight.data), and the layer's transposes made in one launch."""

    def __init__(self, model, i, species, topo, cfg):
        self.inter, self.prod = model.interactions[i], model.products[i]
        self.C, self.first, self.species, self.topo, self.cfg = model.channels, i == 0, species, topo, cfg
        inter, prod = self.inter, self.prod
        up = inter.linear_up
        self.up_w = [_c(up.adapters[str(l)].weight) for l in range(up.lmax + 1)]
        self.up_layout = degree_layout(self.up_w, self.C, up.lmax)
        ml = inter.message_linear
        self.ml_w = [_c(ml.weights[str(l)]) for l in range(ml.lmax + 1)]
        self.ml_layout = path_layout(self.ml_w, ml.counts, self.C, ml.lmax, 1.0 / max(inter.avg_num_neighbors, 1e-8))
        self.pl_wt = [_c(w.t()) for w in prod.linear.blocks()]    # the blocks are transposed views of the weight
        self.pl_layout = degree_layout(self.pl_wt, self.C, prod.target_lmax, self.C ** -0.5)
        self.sc = prod.symmetric_contractions
        self.sc_w = [_c(w) for w in self.sc.slot_weights()]
        self.holder = _SpeciesHolder(species, self.sc.num_elements, shared=True)
        self.Ws = [m.weight.detach() for m in inter.fc if isinstance(m, nn.Linear)]
        if model.radial_basis_scale != 1.0:
            self.Ws[0] = self.Ws[0] * model.radial_basis_scale
        self.Ws = [_c(w) for w in self.Ws]
        made = iter(transposed(self.pl_wt + self.ml_w + ([] if self.first else self.up_w)))
        self.pl_w, self.ml_wt = [next(made) for _ in self.pl_wt], [next(made) for _ in self.ml_w]
        self.up_wt = list(made)

    def _message(self, h, h0, r, Y, mask, table):
        spec, topo = self.inter.spec(), self.topo
        if self.first and self.inter.input_lmax == 0 and tpo.species_form(spec, table.shape[0]):
            self.form, self.xtab = "species", packed_linear_raw(table, self.up_layout, self.up_w)
            self.h3, self.t3 = tpo._mlp_tangent_raw(topo.gate_input(r), self.Ws, self.cfg)
            return tpo._species_fwd_raw(spec, topo, self.xtab, self.species, Y, self.h3, self.Ws[3], mask, topo.gate_rows)
        self.x = packed_linear_raw(h, self.up_layout, self.up_w)
        if tpo._fused_ok(spec, self.x):
            self.form, self.w4s = "fused", tpo._fused_weight(self.Ws[3], spec)
            self.h3, self.t3 = tpo._mlp_tangent_raw(topo.gate_input(r), self.Ws, self.cfg)
            return tpo._fused_fwd_raw(spec, topo, self.x, Y, self.h3, self.w4s, mask, topo.gate_rows)
        self.form = "gates"
        self.gates, self.gdot = radial_gates_tangent(topo.gate_input(r), self.Ws, *self.cfg)
        return tpo._msg_fwd_raw(spec, topo, self.x, Y, self.gates, mask, topo.gate_rows)

    def forward(self, h, h0, r, Y, mask, table):
        self.Y, self.mask = Y, mask
        m = self._message(h, h0, r, Y, mask, table)
        self.message = packed_linear_raw(m, self.ml_layout, self.ml_w)
        del m
        sc = _species_linear(h0, self.inter.self_connection.weights["0"].detach(), self.species)
        out = packed_linear_raw(_fwd_raw(self.sc.spec(), self.message, self.species, self.sc_w, holder=self.holder),
                                self.pl_layout, self.pl_w)
        if out.shape[1] == self.C:
            return out.add_(sc)
        out[:, :self.C] += sc
        return out

    def adjoint(self, dout):
        """Cotangent of the layer's output -> (dh or None, d of its self-connection input or None, dY, dr)."""
        spec, topo = self.inter.spec(), self.topo
        dcon = packed_linear_adjoint_raw(dout, self.pl_layout, self.pl_wt)
        dmsg = _dx_raw(self.sc.spec(), self.message, self.species, self.sc_w, dcon, holder=self.holder)
        del self.message, dcon
        go = packed_linear_adjoint_raw(dmsg, self.ml_layout, self.ml_wt)
        del dmsg
        rows, want = topo.gate_rows, not self.first
        if self.form == "species":
            dx = None
            dY, dr = tpo._species_bwd_raw(spec, topo, self.xtab, self.species, self.Y, self.h3, self.t3, self.Ws[3],
                                          self.mask, go, rows)
        elif self.form == "fused":
            dx, dY, dr = tpo._fused_bwd_raw(spec, topo, self.x, self.Y, self.h3, self.t3, self.w4s, self.mask, go,
                                            (want, True), rows)
        else:
            dx, dY, dr = tpo._msg_bwd_tangent_raw(spec, topo, self.x, self.Y, self.gates, self.gdot, self.mask, go,
                                                  (want, True), rows)
            del self.gates, self.gdot
        if not want:
            return None, None, dY, dr
        ds = dout if dout.shape[1] == self.C else dout[:, :self.C].contiguous()
        ds = _species_linear_adjoint(ds, self.inter.self_connection.weights["0"].detach(), self.species)
        return packed_linear_adjoint_raw(dx, self.up_layout, self.up_wt), ds, dY, dr


@torch.no_grad()
def energy_forces(model, pos, A, batch, edge_src, edge_dst, shifts, cell, topology, owned_mask, graph_energies):
    """(atomic [N], energy64 [graphs], forces [N, 3]), or None where the autograd route has to run.

    graph_energies(selected, batch, cell) sums the owned atomic energies per graph in float64."""
    if not (_plain_context() and _plain_model(model) and _covered(model, pos, A, batch, edge_src, edge_dst, shifts, cell)):
        return None
    N, C = pos.shape[0], model.channels
    pos = pos if pos.is_contiguous() else pos.contiguous()
    check_graph_ids = _graph_ids(batch, cell.shape[0])
    species = model.species_indices(A)
    topo = topology if topology is not None else tpo.Topology(edge_src, edge_dst, N,
                                                              positions=pos if cell.shape[0] == 1 else None)
    if tpo.PAIR_GATES:
        topo.pair_edges(shifts)
    shift = shift_vectors(shifts.to(pos.dtype), cell, batch, edge_src)
    r, n, mask, Y = edge_harmonics_raw(pos, shift, topo, model.max_radius, model.ictd_fix_edge_lmax)
    from mace_ictc.hp.model import SILU_SCALE
    cfg = (float(model.max_radius), int(model.polynomial_cutoff_p), SILU_SCALE)
    table = model.node_embedding.weight.detach().t().contiguous()     # [S, C]
    h = h0 = table.index_select(0, species)
    layers, atomic = [], None
    for i in range(model.num_interaction):
        if i > 0:
            h0 = h if h.shape[1] == C else h[:, :C].contiguous()
            e = edge_linear_raw(h0, model.layer_energy_readouts[i - 1].readout.weight.detach())
            atomic = e if atomic is None else atomic + e
        layer = _Layer(model, i, species, topo, cfg)
        h = layer.forward(h, h0, r, Y, mask, table)
        layers.append(layer)
    last = model.last_layer_energy_readout
    W1, W2, scale = last.linear_1.weight.detach(), last.linear_2.weight.detach(), last.activation._scale
    h0 = h if h.shape[1] == C else h[:, :C].contiguous()
    z = edge_linear_raw(h0, W1)
    e = edge_linear_raw(_silu(0, z, None, None, scale), W2)
    atomic = (e if atomic is None else atomic + e).reshape(N)
    selected = atomic if owned_mask is None else atomic * owned_mask.to(atomic)
    energy64 = graph_energies(selected, batch, cell)

    # adjoint of sum(energy64): one per owned atom
    g = (pos.new_ones(N, 1) if owned_mask is None else owned_mask.to(atomic).reshape(N, 1).contiguous())
    dh = edge_linear_adjoint_raw(_silu(1, z, edge_linear_adjoint_raw(g, W2), None, scale), W1)
    if h.shape[1] != C:
        wide = dh.new_zeros(N, h.shape[1])
        wide[:, :C] = dh
        dh = wide
    del h, h0, z
    cot = []
    for i in range(model.num_interaction - 1, -1, -1):
        dh, ds, dY, dr = layers.pop().adjoint(dh)
        cot.append((dr, dY))
        if i > 0:
            ds += edge_linear_adjoint_raw(g, model.layer_energy_readouts[i - 1].readout.weight.detach())
            dh[:, :C] += ds
    dr, dY = cot[0]
    for a, b in cot[1:-1]:
        dr, dY = dr + a, dY + b
    rest = cot[-1] if len(cot) > 1 else (None, None)
    dvec = edge_harmonics_adjoint_raw(r, n, (dr, dY, *rest), model.ictd_fix_edge_lmax)
    forces = -_vector_adjoint(dvec, topo, N)
    check_graph_ids()
    return atomic, energy64, forces
