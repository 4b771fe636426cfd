"""Rule of the products of few rows (gemm.hip rows_kind): which form takes which sizes."""
import pytest
import torch

from cake_amd.build import GEMM_LIB

pytestmark = pytest.mark.skipif(not GEMM_LIB.exists(), reason="native libraries not built")


def test_rows_kind_lines():
    from cake_amd.ops import gemm as G
    assert G.rows_kind(5, 2048, 2048, False) == 1        # small weights: direct
    assert G.rows_kind(5, 4096, 4096, False) == 1        # 10.3 us, stream 11.5
    assert G.rows_kind(16, 4096, 14336, False) == 2      # large ones: the stream
    assert G.rows_kind(45, 28672, 4096, True) == 2
    assert G.rows_kind(64, 4096, 4096, False) == 0       # tiles
    assert G.rows_kind(65, 28672, 4096, True) == 0
    assert all(G.rows_kind(M, Nv, K, False) != 1 for M in (33, 64) for Nv in (64, 4096)
               for K in (64, 8192))


@pytest.mark.parametrize("M,Nv,K,kind", [
    # us measured as tiles / direct / stream
    (16, 4096, 4096, 2),     # 12.1 / 12.4 / 11.7
    (24, 4096, 4096, 0),     # 12.4 / 14.4 / 15.0
    (16, 6144, 4096, 2),     # 15.7 / 17.9 / 14.3
    (33, 6144, 4096, 0),     # 16.7 / - / 18.3
    (45, 6144, 4096, 0),     # 17.3 / - / 19.1
    (24, 8192, 8192, 2),     # 37.1 / 39.4 / 29.6: parts that start by their strip
    (64, 8192, 8192, 2),     # 39.3 / - / 32.5
    (24, 8192, 16384, 2),    # 65.2 / 75.0 / 46.4
    (24, 10240, 8192, 2),    # 43.3 / 68.2 / 35.2
    (33, 4096, 14336, 0),    # 27.8 / - / 30.1
    (45, 4096, 10928, 0),    # 27.4 / - / 37.6: rows that start amid a line
    (5, 4096, 10928, 2),     # 23.7 / 31.9 / 21.0
    (5, 3072, 2048, 1),      # 9.6 / 6.7 / 8.4
    (24, 5120, 5120, 0),     # 17.2 / 27.6 / 18.3
    (24, 10944, 2048, 0),    # 14.3 / 20.3 / 15.8
    (64, 10240, 8192, 2)])   # 45.5 / - / 41.2
def test_rows_kind_takes_the_measured_best(M, Nv, K, kind):
    from cake_amd.ops import gemm as G
    assert G.rows_kind(M, Nv, K, False) == kind


def test_grouped_rows_stay_out_of_graphs():
    from cake_amd.ops import gemm as G
    assert G.grouped_cfg(78, 64) == G.ROWS and G.grouped_cfg(78, 64, capturing=True) == 4
    assert G.grouped_cfg(64 * 5, 64) == 4


@pytest.mark.parametrize("E,N,K,cfg", [(8, 1024, 2048, 4), (32, 512, 1024, 4), (128, 256, 1024, 4),
                                       (64, 768, 2048, 4), (64, 4096, 3616, 0), (64, 1640, 2048, 0)])
def test_grouped_tiles_of_small_experts(E, N, K, cfg):
    """Between 12 and 24 rows an expert: 128-row tiles only of weights that fill the chip with them."""
    from cake_amd.ops import gemm as G
    assert G.grouped_cfg(16 * E, E, weight=N * K) == cfg
    assert G.grouped_cfg(16 * E, E) == 4 and G.grouped_cfg(24 * E, E, weight=N * K) == 0


@pytest.mark.skipif(torch.cuda.is_available(), reason="makes launches without operands")
@pytest.mark.parametrize("E,N,K,rows", [(1024, 4096, 64, 1500), (512, 8192, 64, 2048),
                                        (1024, 4096, 4096, 4096), (1, 64, 64, 1)])
def test_routed_products_of_any_width_pass_the_checks(E, N, K, rows):
    """Tile lists with more strips than counters are not refused: without a device every call that
    passes the checks ends at its launch, never with an invalid value."""
    from cake_amd.ops import gemm as G
    L, invalid = G._lib(), 1
    tiles = rows // 16 + min(E, rows)
    args = (64, K, 64, K, N * K, 64, N, 64, tiles, 64, 64, 64, N, K, None)
    assert L.cake_gemm_rows_grouped(0, 0, *args) not in (0, invalid)
    assert L.cake_gemm_rows_grouped(0, 1, *args) == invalid   # an epilogue that it does not carry
