"""Edge TP on [channel, magnetic] rows (layout "mul_ir") against the same operator on [magnetic, channel] rows
(tested against the oracle in test_gpu_tp.py): output, first and mixed second derivatives, and a third order, on
channel counts around the 64-channel group, odd row counts and every width of block.  Both layouts round the same
products and sums, up to the contraction of multiply-adds: 2e-6 of the largest value."""
import pytest
import torch

from helpers import rel_err, unit_vectors

import ictc_oracle as orc

pytestmark = pytest.mark.gpu
TOL = 2e-6


def _turn(t, widths, C, to_ir):
    out, off = [], 0
    for w in widths:
        blk = t[:, off:off + w * C]
        blk = blk.reshape(-1, C, w) if to_ir else blk.reshape(-1, w, C)
        out.append(blk.transpose(1, 2).reshape(t.shape[0], -1))
        off += w * C
    return torch.cat(out, 1)


@pytest.mark.parametrize("li,le,lo,C,E", [(0, 1, 1, 1, 3), (1, 1, 1, 17, 5), (2, 2, 2, 64, 257), (2, 2, 2, 65, 33),
                                          (2, 3, 3, 128, 30), (3, 3, 3, 70, 41), (1, 2, 1, 256, 7), (3, 2, 2, 32, 1)])
def test_mul_ir_rows(device, li, le, lo, C, E):
    from ictc_o3 import EdgeTensorProduct
    ops = [EdgeTensorProduct.create(input_lmax=li, edge_lmax=le, output_lmax=lo, channels=C, layout=layout, device=device)
           for layout in ("ir_mul", "mul_ir")]
    with torch.no_grad():
        w = torch.randn_like(ops[0].tp.weight)
        for op in ops:
            op.tp.weight.copy_(w)
    ins = [2 * l + 1 for l in range(li + 1)]
    outs = [2 * l + 1 for l in range(lo + 1) for p in ops[0].paths if p[2] == l]
    g = torch.Generator().manual_seed(C)
    x, gates = torch.randn(E, ops[0].tp.channels * (li + 1) ** 2, generator=g), torch.randn(E, ops[0].gate_width, generator=g)
    sh = torch.cat(orc.direction_harmonics(unit_vectors(E, 4), le), -1).float()
    go = torch.randn(E, ops[0].output_width, generator=g)
    v = [torch.randn(t.shape, generator=g).to(device) for t in (x, sh, gates)]
    u = [torch.randn(t.shape, generator=g).to(device) for t in (x, sh, gates, go)]

    def run(op, mul, third):
        turn = (lambda t, widths, to: _turn(t, widths, C, to)) if mul else (lambda t, widths, to: t)
        leaves = [t.to(device).requires_grad_(True) for t in (x, sh, gates, go)]
        a, b, c, d = leaves
        out = turn(op(turn(a, ins, False), b, c), outs, True)
        first = torch.autograd.grad(out, (a, b, c), d, create_graph=True)
        second = torch.autograd.grad(sum((p * q).sum() for p, q in zip(first, v)), leaves, create_graph=third)
        res = [out, *first, *second]
        if third:
            res += torch.autograd.grad(sum((p * q).sum() for p, q in zip(second, u)), leaves)
        return res
    for third in (False, True):
        for k, (a, b) in enumerate(zip(run(ops[1], True, third), run(ops[0], False, third))):
            assert rel_err(a, b) < TOL, (third, k)


@pytest.mark.parametrize("C", [17, 64, 100])
def test_infinite_gate_of_the_last_channel(device, C):
    """An infinite gate of the scalar path: its products are infinite, and no idle lane makes a NaN of them."""
    from ictc_o3 import EdgeTensorProduct
    E, grads = 5, []
    for layout in ("ir_mul", "mul_ir"):
        op = EdgeTensorProduct.create(input_lmax=1, edge_lmax=1, output_lmax=1, channels=C, layout=layout, device=device)
        assert op.paths[0] == (0, 0, 0)
        x = torch.ones(E, 4 * C, device=device)
        sh = torch.cat(orc.direction_harmonics(unit_vectors(E, 4), 1), -1).float().to(device).requires_grad_(True)
        gates = torch.ones(E, op.gate_width, device=device)
        gates[:, C - 1] = float("inf")
        out = op(x, sh, gates)
        grads.append(torch.autograd.grad(out, sh, torch.ones_like(out))[0])
    assert bool(torch.isinf(grads[0][:, 0]).all()) and bool(torch.isfinite(grads[0][:, 1:]).all())
    # (of the row's finite values: the layouts' sums in another order)
    assert torch.allclose(grads[1], grads[0], rtol=1e-5, atol=1e-5 * C)
