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
