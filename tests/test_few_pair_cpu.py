"""Which blocks of up to eight rows run their output and gated products as gemm_few.hip has them."""
import pytest

from cake_amd.ops import gemm as G


@pytest.mark.parametrize("M,H,K,inter,takes", [
    (5, 2048, 2048, 8192, True), (8, 3072, 4096, 14336, True), (9, 2048, 2048, 8192, False), (5, 4096, 4096, 14336, False),
    # narrow rows: as long as there are not many of them
    (5, 256, 256, 3072, True), (5, 256, 256, 3080, False), (5, 256, 256, 32768, False), (1, 64, 64, 131072, False),
    (5, 1016, 1024, 12192, True), (5, 1016, 1024, 12208, False), (5, 1024, 1024, 16384, True), (5, 32, 32, 64, True)])
def test_the_line(M, H, K, inter, takes):
    assert G.few_pair(M, H, K, inter) == takes


def test_the_librarys_plan_is_its_own(monkeypatch):
    """A measured plan that names the library GEMM stands, as for every product, where no form of few rows does."""
    M, H, K, inter = 3, 64, 32, 128
    assert G.few_pair(M, H, K, inter)
    monkeypatch.setattr(G, "rows_kind", lambda *a: 0)
    monkeypatch.setattr(G, "resolve", lambda m, n, k, epi, *a, **kw: (G.LIB if epi == "swiglu" else 4, 1))
    assert not G.few_pair(M, H, K, inter)


def test_products_of_the_pair_have_no_form():
    """A native run forms no plan for products that the pair's kernels run, and holds no workspace for them."""
    from cake_amd.ops import llama_rows as L
    forms, floats, left = L._forms(((5, 3072, 2048, "store", True), None, None, (5, 2048, 8192, "resid32", True)), False)
    assert [(f.kind, f.cfg, f.splits, f.slabs) for f in forms[1:3]] == [(0, 0, 0, 0)] * 2 and forms[0].slabs
