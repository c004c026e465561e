"""energy_and_forces(training=False) without autograd (mace_ictc/hp/direct.py) against the autograd route of the same
call, which the oracle tests cover: every message form, 1 to 3 layers, batches, owned masks, channel counts with and
without the species kernels, and systems on both sides of the table and row-split rules.  Both run the same kernels;
sums of two cotangents may round in another order, so 2e-6 of the largest value.  Where the graph could be observed
the call takes the autograd route."""
import pytest
import torch

from helpers import rel_err
from model_helpers import build_graph, fcc_cells

pytestmark = pytest.mark.gpu
ZS = (1, 6, 7, 8, 9)


def _system(device, S, cells, ncell, cutoff=4.5):
    pos, Z, batch, cell = fcc_cells(ncell, 0.1, 0.3, 3, S, cells=cells, atomic_numbers=ZS[:S])
    src, dst, sh = build_graph(pos, batch, cell, cutoff)
    return [t.to(device) for t in (pos.float(), Z, batch, src, dst, sh.float(), cell.float())]


def _model(device, S, **kw):
    from mace_ictc.hp import create_model
    torch.manual_seed(5)
    return create_model(atomic_numbers=ZS[:S], cutoff=4.5, avg_num_neighbors=40.0, device=device, **kw)


@pytest.mark.parametrize("kw,S,cells,ncell,masked", [
    (dict(channels=64, lmax=2), 3, 1, 2, False),                        # species form, then materialised gates
    (dict(channels=64, lmax=2), 5, 2, 2, True),                         # fused first layer, batch, owned mask
    (dict(channels=128, lmax=2, edge_lmax=3), 4, 1, 3, True),           # degree-3 edges
    (dict(channels=32, lmax=1, num_interactions=3, correlation=2), 5, 1, 2, False),
    (dict(channels=48, lmax=1, num_interactions=1), 2, 3, 2, False),
    (dict(channels=16, lmax=0, edge_lmax=1), 3, 1, 2, False),
    (dict(channels=64, lmax=2, edge_lmax=3, correlation=1), 2, 1, 9, False)])
def test_direct_matches_autograd(device, kw, S, cells, ncell, masked, monkeypatch):
    from mace_ictc.hp import direct, energy_and_forces
    model, args = _model(device, S, **kw), _system(device, S, cells, ncell)
    mask = (torch.rand(args[0].shape[0], device=device) > 0.3) if masked else None
    calls = []
    inner = direct.energy_forces
    monkeypatch.setattr(direct, "energy_forces", lambda *a: calls.append(inner(*a)) or calls[-1])
    got = energy_and_forces(model, *args, owned_mask=mask)
    assert calls[-1] is not None
    again = energy_and_forces(model, *args, owned_mask=mask)
    monkeypatch.setattr(direct, "DIRECT", False)
    ref = energy_and_forces(model, *args, owned_mask=mask)
    assert calls[-1] is None
    for k in ("energy", "forces", "atomic_energy"):
        assert got[k].dtype == ref[k].dtype and got[k].shape == ref[k].shape and not got[k].requires_grad
        assert rel_err(got[k], ref[k]) < 2e-6, k
        assert torch.equal(got[k], again[k]), k


def test_observable_graphs_take_the_autograd_route(device):
    from mace_ictc.hp import direct, energy_and_forces
    from mace_ictc.hp.runtime import _graph_energies
    model, args = _model(device, 3, channels=16, lmax=1), _system(device, 3, 1, 2)

    def direct_runs(a=args):
        return direct.energy_forces(model, *a, None, None, _graph_energies) is not None
    assert direct_runs()
    ref = energy_and_forces(model, *args)["forces"]
    seen = []
    handle = model.interactions[1].register_forward_hook(lambda *a: seen.append(1))
    assert not direct_runs()
    assert rel_err(energy_and_forces(model, *args)["forces"], ref) < 2e-6 and seen
    handle.remove()
    pos = args[0].clone().requires_grad_(True)
    grads = []
    pos.register_hook(lambda g: grads.append(g))
    energy_and_forces(model, pos, *args[1:])
    assert grads and not direct_runs([pos, *args[1:]])
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
        assert not direct_runs()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not direct_runs()
    up = model.interactions[1].linear_up.adapters["0"]
    torch.nn.utils.parametrize.register_parametrization(up, "weight", torch.nn.Identity())
    assert not direct_runs()
    assert rel_err(energy_and_forces(model, *args)["forces"], ref) < 2e-6
    torch.nn.utils.parametrize.remove_parametrizations(up, "weight")
    assert direct_runs()
    assert not direct_runs([*args[:3], *(t[:0] for t in args[3:6]), args[6]])     # no edges
    single, one = _model(device, 1, channels=16, lmax=1), _system(device, 1, 1, 2)
    assert direct.energy_forces(single, *one, None, None, _graph_energies) is None  # a one-row species table
    with pytest.raises(ValueError, match="without compact mapping"):
        energy_and_forces(model, args[0], torch.full_like(args[1], 17), *args[2:])
