"""energy_and_forces(training=False) without autograd reads the weights as they are at each call: a write in place,
through .data (as weight averaging does), a new storage, and a weight kept in transposed storage.  The reference is
the autograd route of a fresh copy of the model, which has kept nothing from earlier calls."""
import copy

import pytest
import torch

from helpers import rel_err
from model_helpers import build_graph, fcc_cells

pytestmark = pytest.mark.gpu
ZS = (1, 6, 7, 8, 9)


def _system(device, S):
    pos, Z, batch, cell = fcc_cells(2, 0.1, 0.3, 3, S, cells=1, atomic_numbers=ZS[:S])
    src, dst, sh = build_graph(pos, batch, cell, 4.5)
    return [t.to(device) for t in (pos.float(), Z, batch, src, dst, sh.float(), cell.float())]


def _model(device, S):
    from mace_ictc.hp import create_model
    torch.manual_seed(5)
    return create_model(atomic_numbers=ZS[:S], cutoff=4.5, avg_num_neighbors=40.0, device=device, channels=64, lmax=2)


def _in_place(p, new):
    with torch.no_grad():
        p.copy_(new)


def _through_data(p, new):
    p.data.copy_(new)


def _new_storage(p, new):
    p.data = new


def _check(monkeypatch, model, args, what):
    from mace_ictc.hp import direct, energy_and_forces
    got = energy_and_forces(model, *args)
    monkeypatch.setattr(direct, "DIRECT", False)
    ref = energy_and_forces(copy.deepcopy(model), *args)
    monkeypatch.setattr(direct, "DIRECT", True)
    for k in ("energy", "forces", "atomic_energy"):   # two routes of the same kernels: sums in another order
        assert rel_err(got[k], ref[k]) < 2e-6, (what, k)
    return got["forces"]


@pytest.mark.parametrize("change", [_in_place, _through_data, _new_storage])
@pytest.mark.parametrize("transposed", [False, True])
def test_last_radial_weight_of_the_fused_message(device, monkeypatch, change, transposed):
    model, args = _model(device, 5), _system(device, 5)      # five species: the first layer's message is fused
    lin = model.interactions[0].fc[-1]
    if transposed:
        lin.weight = torch.nn.Parameter(lin.weight.detach().t().contiguous().t())
    before = _check(monkeypatch, model, args, "as built")
    change(lin.weight, (1.5 * lin.weight.detach()).clone(memory_format=torch.preserve_format))
    moved = rel_err(_check(monkeypatch, model, args, change.__name__), before)
    assert moved > 1e-2


@pytest.mark.parametrize("change", [_in_place, _through_data, _new_storage])
@pytest.mark.parametrize("S", [3, 5])
def test_node_embedding(device, monkeypatch, change, S):
    model, args = _model(device, S), _system(device, S)
    w = model.node_embedding.weight
    before = _check(monkeypatch, model, args, "as built")
    change(w, -0.5 * w.detach())
    moved = rel_err(_check(monkeypatch, model, args, change.__name__), before)
    assert moved > 1e-2
