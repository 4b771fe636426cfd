"""Tiles of grouped products by rows an expert, weights and width of the rows."""
import pytest

from cake_amd.ops import gemm as G


@pytest.mark.parametrize("E,F,W", [(64, 3648, 4096), (128, 768, 2048), (8, 2048, 1032), (16, 1024, 1024), (8, 512, 64)])
def test_rule(E, F, W):
    """Of wide rows the stream form up to four rows an expert, up to eight of fewer weights, then 128-row tiles; a capture
    takes no stream form; narrow rows are where they were without a width."""
    for mean in (1, 4, 5, 8, 9, 23, 24, 63, 64, 500):
        for capturing in (False, True):
            cfg = G.grouped_cfg(mean * E, E, capturing, F * W, W)
            if W <= 1024:
                assert cfg == G.grouped_cfg(mean * E, E, capturing, F * W)
            elif not capturing and mean <= (8 if E * F * W < 220e6 else 4):
                assert cfg == G.ROWS
            elif capturing and mean <= 4:
                assert cfg == 0
            else:
                assert cfg == (0 if mean < 64 else G.BY_LIST)
