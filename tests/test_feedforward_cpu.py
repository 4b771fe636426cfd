"""Layout of the feed-forwards' weights (models/hybrid/feedforward.py)."""
import pytest
import torch

from cake_amd.models.hybrid import feedforward as F
from cake_amd.models.hybrid.config import DenseMlp, ExpertsMlp


@pytest.mark.parametrize("ff,cols", [(8, 8), (13, 16), (72, 72), (992, 992), (1000, 1024), (1056, 1088),
                                     (1824, 1856), (3616, 3648), (4096, 4096)])
@pytest.mark.parametrize("experts", [0, 3])
def test_rows_are_whole_lines_where_that_adds_little(ff, cols, experts):
    """Down rows (and the activations they read) end on 128-byte lines; what is added is zero."""
    W = 16
    assert F.columns(ff) == cols
    m = ExpertsMlp(ff, experts, 2) if experts else DenseMlp(ff, act="relu2", bias=True)
    shapes = F.tensor_shapes(m, W)
    w = F.load(m, lambda n, dtype=torch.bfloat16: torch.ones(shapes.get(n.split("mlp.")[-1], (W,)), dtype=dtype),
               "l0.", type("C", (), {"width_padded": W}), "cpu", torch.bfloat16)
    assert w.up.shape[-2:] == (cols, W) and w.down.shape[-2:] == (W, cols)
    assert bool((w.up[..., :ff, :] == 1).all()) and not bool(w.up[..., ff:, :].any())
    assert bool((w.down[..., :ff] == 1).all()) and not bool(w.down[..., ff:].any())
