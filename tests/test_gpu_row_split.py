"""Message sums over rows split over 1, 2 or 4 waves (sum_parts): forward, first adjoint and mixed second
derivative against the float64 oracle on both sides of each row count where the split changes, with empty rows,
one row of several 64-edge chunks (uneven shares) and a shuffled row order.  Tolerance 1e-5 relative (max-norm),
as the message tests: FP32 sums of up to 600 terms."""
import pytest
import torch

import ictc_oracle as orc
from helpers import rel_err, unit_vectors

pytestmark = pytest.mark.gpu
TOL = 1e-5


@pytest.mark.parametrize("N,C,li,le,lo", [(1, 16, 2, 2, 2), (3, 70, 1, 2, 2), (2047, 16, 1, 1, 1), (2048, 16, 1, 1, 1),
                                          (4096, 16, 1, 1, 1), (8191, 16, 1, 1, 1), (8192, 8, 1, 1, 1),
                                          (16384, 8, 0, 1, 1)])
def test_split_rows(device, N, C, li, le, lo):
    from ictc_o3 import PackedGraphMessage
    from ictc_o3.ops import tensor_product as tpo
    op = PackedGraphMessage.create(channels=C, input_lmax=li, edge_lmax=le, output_lmax=lo, device=device)
    g = torch.Generator().manual_seed(N)
    E = 2 * N + 605
    src, dst = torch.randint(0, N, (E,), generator=g), torch.randint(0, N, (E,), generator=g)
    dst[:301] = N // 2        # a receiver and a source with several chunks
    src[300:601] = N // 3
    feats = torch.randn(N, C * (li + 1) ** 2, generator=g, dtype=torch.float64)
    sh = torch.cat(orc.direction_harmonics(unit_vectors(E, N + 1), le), -1)
    gates = torch.randn(E, op.gate_width, generator=g, dtype=torch.float64)
    go = torch.randn(N, op.output_width, generator=g, dtype=torch.float64)
    v = [torch.randn(t.shape, generator=g, dtype=torch.float64) for t in (feats, sh, gates)]

    def run(tensors, cot, fn):
        xs = [t.clone().requires_grad_(True) for t in tensors]
        cot = cot.clone().requires_grad_(True)
        out = fn(*xs)
        grads = torch.autograd.grad(out, xs, cot, create_graph=True)
        second = torch.autograd.grad(sum((a * b.to(a)).sum() for a, b in zip(grads, v)), xs + [cot])
        return [out, *grads, *second]

    ref = run((feats, sh, gates), go, lambda a, b, c: orc.message_packed(a, b, c, src, dst, None, li, le, lo, C))
    topo = tpo.Topology(src.to(device), dst.to(device), N)
    topo.src_rows = torch.randperm(N, generator=g).int().to(device)
    topo.dst_rows = torch.randperm(N, generator=g).int().to(device)
    got = run([t.float().to(device) for t in (feats, sh, gates)], go.float().to(device),
              lambda a, b, c: op(a, b, c, topo.src, topo.dst, topology=topo))
    for name, a, b in zip(("out", "dx", "dsh", "dg", "d2x", "d2sh", "d2g", "d2go"), got, ref):
        assert rel_err(a, b) < TOL, name
