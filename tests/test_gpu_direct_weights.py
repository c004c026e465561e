"""energy_and_forces(training=False) without autograd reads the weights as they are at each call: a write in place,
through .data (as weight averaging does), a new storage, and a weight kept in transposed storage.  The reference is
the autograd route of a fresh copy of the model, which has kept nothing from earlier calls."""
import copy
import gc

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


WEIGHTS = {"linear_up": lambda m: m.interactions[1].linear_up.adapters["1"].weight,
           "message_linear": lambda m: m.interactions[1].message_linear.weights["2"],
           "product": lambda m: m.products[0].linear.weight,
           "self_connection": lambda m: m.interactions[1].self_connection.weights["0"],
           "contraction": lambda m: m.products[0].symmetric_contractions.slot_weights()[0],
           "radial": lambda m: m.interactions[1].fc[2].weight}


@pytest.mark.parametrize("change", [_in_place, _through_data, _new_storage])
@pytest.mark.parametrize("name", WEIGHTS)
def test_other_weights(device, monkeypatch, change, name):
    model, args = _model(device, 3), _system(device, 3)
    w = WEIGHTS[name](model)
    before = _check(monkeypatch, model, args, "as built")
    change(w, -0.5 * w.detach() + 0.1)
    moved = rel_err(_check(monkeypatch, model, args, change.__name__), before)
    assert moved > 1e-4


def test_calls_keep_no_copies_of_weights(device):
    from ictc_o3.ops import linear
    from mace_ictc.hp import energy_and_forces
    model, args = _model(device, 3), _system(device, 3)
    energy_and_forces(model, *args)
    linear._operand_cache.clear()
    gc.collect()
    torch.cuda.synchronize()
    held = torch.cuda.memory_allocated()
    for _ in range(3):
        energy_and_forces(model, *args)
    assert not linear._operand_cache and torch.cuda.memory_allocated() == held


@pytest.mark.parametrize("shapes", [[(1, 1)], [(33, 31)], [(64, 5), (0, 7), (128, 2176), (32, 32), (5, 0), (1, 200)],
                                    [(k % 40 + 1, 70 - k) for k in range(65)]])    # 64 matrices a launch
def test_transposed(device, shapes):
    from ictc_o3.ops.linear import transposed
    mats = [torch.randn(*s, device=device) for s in shapes]
    for m, t in zip(mats, transposed(mats)):
        assert t.is_contiguous() and t.data_ptr() % 16 == 0 and torch.equal(t, m.t())
