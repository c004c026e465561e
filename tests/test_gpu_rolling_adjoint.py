"""One-pass source-owned adjoints whose edge rows load into the registers that the previous edge has read
(msg_bwd_src kernels), against the separate kernels of the same quantities: the receiver-owned pass (dsh, dr or
dgates) and the feature-gradient pass (dx), which share neither loops nor generated contraction with them.
Every degree triple's register class, path weights, one and two channel groups, sources of 0, 1, 63, 64, 65 and
130 edges (chunk edges), masks, shared gate rows and out-of-range ids.

Tolerances, relative in the max norm: dx sums up to 130 edges of at most 23 * 49 products each, dsh and dr reduce
up to 23 * 128 products over lanes; reassociated FP32 sums of n terms differ by about sqrt(n) eps/2 = 6e-6 at
n = 1e4 in the worst of these, 1e-5 as in the message tests."""
import pytest
import torch

from helpers import rel_err
from test_gpu_message import _graph

pytestmark = pytest.mark.gpu
TOL = 1e-5
LENGTHS = (0, 1, 63, 64, 65, 130)


def _case(device, C, li, le, lo, weighted):
    from ictc_o3.ops import tensor_product as tpo
    N = 40
    E = 4 * N + sum(LENGTHS)
    f64, sh64, g64, src, dst, m64 = _graph(N, E, C, li, le, lo, 7 + 100 * li + 10 * le + lo, mask=True)
    src = torch.cat([torch.full((n,), 3 * k) for k, n in enumerate(LENGTHS)] + [src[:4 * N] % 20 + 20])
    src[-9], dst[-5], dst[70] = N + 3, -1, N
    spec = tpo.make_spec(li, le, lo, C)
    if weighted:
        w = torch.rand(spec.num_paths, C, generator=torch.Generator().manual_seed(3)) + 0.5
        spec = tpo.make_spec(li, le, lo, C, w.to(device))
    topo = tpo.Topology(src.to(device), dst.to(device), N)
    gen = torch.Generator(device=device).manual_seed(11)
    x, sh, g, m = (t.float().to(device) for t in (f64, sh64, g64, m64))
    go = torch.randn(N, spec.out_components * C, device=device, generator=gen)
    return tpo, spec, topo, x, sh, g, m, go, gen


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("C,li,le,lo", [(64, 2, 2, 2), (70, 2, 2, 2), (16, 1, 1, 1), (32, 0, 2, 2), (64, 1, 3, 3),
                                        (96, 3, 3, 1), (128, 2, 3, 3), (64, 3, 3, 3), (48, 2, 2, 3), (8, 3, 0, 3)])
def test_tangent_adjoint(device, C, li, le, lo, weighted):
    tpo, spec, topo, x, sh, g, m, go, gen = _case(device, C, li, le, lo, weighted)
    E = sh.shape[0]
    rows = torch.randint(0, E // 2, (E,), device=device, generator=gen, dtype=torch.int32)
    gates, gdot = g[:E // 2].contiguous(), torch.randn(E // 2, g.shape[1], device=device, generator=gen)
    dx, dsh, dr = tpo._msg_bwd_tangent_raw(spec, topo, x, sh, gates, gdot, m, go, (True, True), rows)
    none, dsh0, dr0 = tpo._msg_bwd_tangent_raw(spec, topo, x, sh, gates, gdot, m, go, (False, True), rows)
    dx0 = tpo._msg_bwd_raw(spec, topo, x, sh, gates[rows.long()], m, go, (True, False, False))[0]
    assert none is None
    for a, b in ((dx, dx0), (dsh, dsh0), (dr, dr0)):
        assert rel_err(a, b) < TOL
    only_x, no_sh, dr1 = tpo._msg_bwd_tangent_raw(spec, topo, x, sh, gates, gdot, m, go, (True, False), rows)
    assert no_sh is None and torch.equal(only_x, dx) and rel_err(dr1, dr0) < TOL
    out = (topo.src < 0) | (topo.src >= 40) | (topo.dst < 0) | (topo.dst >= 40)
    assert out.sum() == 3 and torch.count_nonzero(dr[out]) == 0 and torch.count_nonzero(dsh[out]) == 0


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("C,li,le,lo", [(64, 2, 2, 2), (70, 2, 2, 2), (16, 1, 1, 1), (32, 0, 2, 2), (64, 1, 3, 3),
                                        (96, 3, 3, 1), (128, 2, 3, 3), (64, 3, 3, 3), (48, 2, 2, 3), (8, 3, 0, 3)])
def test_adjoint(device, C, li, le, lo, weighted):
    tpo, spec, topo, x, sh, g, m, go, gen = _case(device, C, li, le, lo, weighted)
    dx, dsh, dg = tpo._msg_bwd_raw(spec, topo, x, sh, g, m, go, (True, True, True))
    _, dsh0, dg0 = tpo._msg_bwd_raw(spec, topo, x, sh, g, m, go, (False, True, True))
    dx0 = tpo._msg_bwd_raw(spec, topo, x, sh, g, m, go, (True, False, False))[0]
    for a, b in ((dx, dx0), (dsh, dsh0), (dg, dg0)):
        assert rel_err(a, b) < TOL
    held = torch.randn(g.shape, device=device, generator=gen)
    into = held.clone()
    tpo._msg_bwd_raw(spec, topo, x, sh, g, m, go, (True, True, True), dg_into=into)
    assert torch.equal(into, held + dg)
    out = (topo.src < 0) | (topo.src >= 40) | (topo.dst < 0) | (topo.dst >= 40)
    assert torch.count_nonzero(dg[out]) == 0 and torch.count_nonzero(dsh[out]) == 0
    assert torch.count_nonzero(dx[0]) == 0        # the source without edges
