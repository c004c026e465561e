"""Symmetric contraction on per-species coefficient tables (ictc_sc_table_*).

Every mode against the per-node kernels (tested against the oracle in test_gpu_sc.py) on node counts around the
tile (3 or 4 nodes a wave, 4 waves a block) and chunk (32 or more nodes) sizes, with empty species, out-of-range ids and channel counts
that leave idle lanes; both forms round sums of the same FP32 products, so 1e-5 of the largest value holds each.
The route taken by size is compared once with the float64 oracle.
"""
import pytest
import torch

from helpers import rel_err
from test_gpu_sc import _oracle_packed, _oracle_weights, _packed, _setup

pytestmark = pytest.mark.gpu
TOL = 1e-5


@pytest.mark.parametrize("lmax,lt,C,N,S", [(2, 2, 64, 1, 1), (2, 2, 70, 333, 3), (3, 1, 17, 47, 2), (3, 1, 64, 129, 1),
                                           (3, 2, 64, 16, 2), (3, 2, 100, 2100, 7),
                                           # 64 species a step of the tile search: its edges, and more nodes than one tile
                                           (2, 2, 64, 900, 63), (3, 1, 64, 500, 64), (2, 2, 16, 3000, 200)])
def test_table_kernels_match_per_node(device, lmax, lt, C, N, S, monkeypatch):
    from ictc_o3.ops import symmetric_contraction as sco
    mod, x64, species = _setup(device, lmax, lt, 3, C, N, S, 5)
    species[N // 2:N // 2 + 3] = S + 4        # out-of-range ids: zero rows, no weight gradient
    species[N // 3] = -1
    if S > 2:
        species[species == 1] = 2             # a species without nodes
    spec, ws = mod.spec(), [w.detach() for w in mod.slot_weights()]
    x, sp = _packed(x64, lmax).float().to(device), species.to(device)
    g = torch.Generator().manual_seed(6)
    go = torch.randn(N, spec.no * C, generator=g).to(device)
    h = torch.randn(N, spec.nx * C, generator=g).to(device)
    holder = sco._SpeciesHolder(sp, S)

    def run():
        return ([sco._fwd_raw(spec, x, sp, ws, t, holder=holder) for t in (None, h)]
                + [sco._dx_raw(spec, x, sp, ws, go, t, holder=holder) for t in (None, h)]
                + sco._dw_raw(spec, x, holder.species_csr(), go) + sco._dw_raw(spec, x, holder.species_csr(), go, h))
    monkeypatch.setattr(sco, "_use_table", lambda spec, N, weights=False: False)
    ref = run()
    monkeypatch.setattr(sco, "_use_table", lambda spec, N, weights=False: True)
    got = run()
    for k, (a, b) in enumerate(zip(got, ref)):
        assert rel_err(a, b) < TOL, k
    assert all(torch.equal(a, b) for a, b in zip(got, run()))


@pytest.mark.parametrize("lmax,lt,C,N,S", [(3, 2, 128, 2050, 10), (2, 2, 16, 32770, 3)])
def test_table_route_matches_oracle(device, lmax, lt, C, N, S):
    from ictc_o3.ops import symmetric_contraction as sco
    mod, x64, species = _setup(device, lmax, lt, 3, C, N, S, 8)
    assert sco._use_table(mod.spec(), N)
    W = _oracle_weights(mod)
    ref = _oracle_packed(x64[:256], species[:256], W, lmax, lt, 3, C)
    out = mod.contract(_packed(x64, lmax).float().to(device), species.to(device))
    assert rel_err(out[:256], ref) < TOL
