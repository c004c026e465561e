"""Which contractions take the per-species coefficient tables (ops/symmetric_contraction._use_table), from sizes alone."""
import pytest

from ictc_o3.ops import symmetric_contraction as sco


@pytest.mark.parametrize("lmax,lt,C,N,S,table,weights", [
    (3, 2, 128, 8191, 10, True, True), (3, 2, 128, 8191, 89, True, True), (2, 2, 64, 131072, 89, True, True),
    # few nodes of each species: the table and the pair sums cost more than they save
    (3, 2, 128, 8191, 250, False, False), (3, 1, 64, 8191, 250, False, False), (2, 2, 64, 131072, 4000, False, False),
    (2, 2, 64, 131072, 1000, False, True),
    # few nodes in all; a shape without tables
    (3, 2, 64, 2048, 4, False, False), (2, 2, 64, 8000, 4, False, True), (2, 1, 64, 131072, 4, False, False),
    # more species or nodes than the table kernels take
    (2, 2, 64, 65536 * 512, 65536, False, False), (3, 2, 64, 2 ** 31, 4, False, False)])
def test_rule(lmax, lt, C, N, S, table, weights):
    spec = sco.ScSpec(lmax, lt, 3, C, S)
    assert sco._use_table(spec, N) == table and sco._use_table(spec, N, weights=True) == weights


@pytest.mark.parametrize("lmax,lt,C,N,alone", [(3, 2, 64, 4096, True), (3, 1, 64, 8191, False), (3, 1, 128, 5120, True),
                                               (2, 2, 64, 32768, False), (2, 2, 64, 65536, True), (2, 2, 100, 20000, False)])
def test_the_order_is_made_for_the_tables_alone_where_it_pays(lmax, lt, C, N, alone):
    spec = sco.ScSpec(lmax, lt, 3, C, 4)
    assert sco._use_table(spec, N)
    assert sco._order_pays(spec, N, sco._SpeciesHolder(None, 4)) == alone
    assert sco._order_pays(spec, N, sco._SpeciesHolder(None, 4, weight_gradients=True))
    assert sco._order_pays(spec, N, sco._SpeciesHolder(None, 4, shared=True)) == (alone or C in (64, 128))
    made = sco._SpeciesHolder(None, 4)
    made._csr = object()
    assert sco._order_pays(spec, N, made)
