"""energy_and_forces(training=False) without autograd at the widest degree, and what it refuses as the autograd route
does: graph ids outside the batch (every kernel that reads them checks them, so nothing is read out of range before the call raises), and edge
shifts that are not one per edge (refused on the host before a launch)."""
import pytest
import torch

from model_helpers import build_graph, fcc_cells

pytestmark = pytest.mark.gpu


def _batch(device, cells):
    from mace_ictc.hp import create_model
    torch.manual_seed(5)
    model = create_model(atomic_numbers=(1, 6, 8), cutoff=4.5, device=device, channels=16, lmax=1)
    pos, Z, batch, cell = fcc_cells(2, 0.1, 0.3, 3, 3, cells=cells, atomic_numbers=(1, 6, 8))
    src, dst, sh = build_graph(pos, batch, cell, 4.5)
    return model, [t.to(device) for t in (pos.float(), Z, batch, src, dst, sh.float(), cell.float())]


@pytest.mark.parametrize("cells,wrong", [(2, -1), (2, 2), (70, 70)])    # 70 graphs: the sum looks at the order too
@pytest.mark.parametrize("isolated", [True, False])
def test_graph_ids_out_of_range(device, cells, wrong, isolated):
    from mace_ictc.hp import energy_and_forces
    model, (pos, Z, batch, src, dst, sh, cell) = _batch(device, cells)
    atom = 0 if wrong < 0 else pos.shape[0] - 1
    keep = (src != atom) & (dst != atom) if isolated else torch.ones_like(src, dtype=torch.bool)
    graph = (src[keep], dst[keep], sh[keep], cell)
    energy_and_forces(model, pos, Z, batch, *graph)
    bad = batch.clone()
    bad[atom] = wrong
    with pytest.raises(ValueError, match="Graph ids"):
        energy_and_forces(model, pos, Z, bad, *graph)
    energy_and_forces(model, pos, Z, batch, *graph)


def test_one_graph_ignores_the_ids(device):
    from mace_ictc.hp import energy_and_forces
    model, args = _batch(device, 1)
    ref = energy_and_forces(model, *args)
    got = energy_and_forces(model, *args[:2], args[2] + 5, *args[3:])
    assert torch.equal(got["forces"], ref["forces"]) and torch.equal(got["energy"], ref["energy"])


@pytest.mark.parametrize("paired", [True, False])      # pairing the edges looks at the shifts as well
@pytest.mark.parametrize("more", [-1, 1])
def test_shifts_one_per_edge(device, monkeypatch, paired, more):
    from ictc_o3.ops import tensor_product as tpo
    from mace_ictc.hp import energy_and_forces
    model, args = _batch(device, 1)
    shifts = args[5][:-1] if more < 0 else torch.cat([args[5], args[5][:1]])
    monkeypatch.setattr(tpo, "PAIR_GATES", paired)
    with pytest.raises(ValueError, match=r"\[E, 3\]"):
        energy_and_forces(model, *args[:5], shifts, args[6])


@pytest.mark.parametrize("S", [3, 5])      # the first layer's message: gates materialised (no species form at edge degree 3)
def test_widest_degree_matches_autograd(device, monkeypatch, S):
    """lmax 3 and one layer (the contraction onto degree 3, which more layers need, is not compiled)."""
    from helpers import rel_err
    from mace_ictc.hp import create_model, direct, energy_and_forces
    torch.manual_seed(5)
    zs = (1, 6, 7, 8, 9)[:S]
    model = create_model(lmax=3, num_interactions=1, atomic_numbers=zs, cutoff=4.5, device=device)
    pos, Z, batch, cell = fcc_cells(3, 0.1, 0.3, 3, S, cells=1, atomic_numbers=zs)
    src, dst, sh = build_graph(pos, batch, cell, 4.5)
    args = [t.to(device) for t in (pos.float(), Z, batch, src, dst, sh.float(), cell.float())]
    got = energy_and_forces(model, *args)
    monkeypatch.setattr(direct, "DIRECT", False)
    ref = energy_and_forces(model, *args)
    for k in ("energy", "forces", "atomic_energy"):   # two routes of the same kernels: sums in another order
        assert rel_err(got[k], ref[k]) < 2e-6, k
