"""The species order kept between calls (ops/linear.species_order): one thread's read is not mixed with another's
write, another stream and a captured stream make their own."""
import pytest
import torch

from helpers import rel_err


def test_memo_replaced_between_reads(monkeypatch):
    """Another thread replaces the memo while this one compares it: the order returned is that of its own species."""
    from ictc_o3.ops import linear as lin

    class Order:
        def __init__(self, species, S):
            self.species = species
    monkeypatch.setattr(lin, "SpeciesOrder", Order)
    monkeypatch.setattr(lin.nat, "stream_of", lambda t: 0)
    a, b = torch.zeros(4, dtype=torch.long), torch.ones(4, dtype=torch.long)

    class Replaced(tuple):
        def __getitem__(self, i):
            if i == 1:      # after the key has been compared
                lin._order_memo = other
            return tuple.__getitem__(self, i)
    monkeypatch.setattr(lin, "_order_memo", None)
    lin.species_order(b, 3)
    other = lin._order_memo
    first = lin.species_order(a, 3)
    lin._order_memo = Replaced(lin._order_memo)
    assert lin.species_order(a, 3) is first and first.species is a


@pytest.mark.gpu
def test_each_stream_makes_its_own(device):
    from ictc_o3.ops import linear as lin
    sp = torch.randint(0, 5, (1000,), device=device)
    order = lin.species_order(sp, 5)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        other = lin.species_order(sp, 5)
        assert other is not order and lin.species_order(sp, 5) is other
    torch.cuda.synchronize()
    assert torch.equal(other.perm, order.perm) and torch.equal(other.off, order.off)


@pytest.mark.gpu
def test_captured_stream_makes_its_own(device):
    from ictc_o3.ops import linear as lin
    g = torch.Generator(device=device).manual_seed(2)
    sp = torch.randint(0, 5, (700,), device=device, generator=g)
    x, W = torch.randn(700, 64, device=device, generator=g), torch.randn(5, 64, 64, device=device, generator=g)
    with torch.no_grad():
        lin.species_linear(x, W, sp)      # the memo holds this species tensor's order
        torch.cuda.synchronize()
        memo = lin._order_memo
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = lin.species_linear(x, W, sp)
        assert lin._order_memo is memo
        for k in range(4):
            x.copy_(torch.randn(700, 64, device=device, generator=g))
            sp.copy_(torch.randint(0, 5, (700,), device=device, generator=g))
            graph.replay()
            torch.cuda.synchronize()
            other = torch.randint(0, 5, (700,), device=device, generator=g)      # replaces the memo between replays
            lin.species_linear(x, W, other)
            ref = torch.einsum("noi,ni->no", W.double().cpu()[sp.cpu()], x.double().cpu())
            assert rel_err(out, ref) < 1e-5
