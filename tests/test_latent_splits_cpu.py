"""Splits of latent decode by the sequences of a step."""
from types import SimpleNamespace

import pytest

from cake_amd.models.hybrid import model as H


@pytest.mark.parametrize("nsplit", [n for _, n in H.SPLITS])
@pytest.mark.parametrize("heads", [1, 16, 17, 128])
def test_splits(nsplit, heads):
    """As many as the keys have tiles for, a power of two, halved while the workgroups are more than CUs; one at least.
    Short sequences beside a long one count by their keys."""
    groups = -(-heads // 16)
    for B in (1, 2, 3, 8, 13, 16, 17, 255, 256, 257, 4096):
        n = H.latent_splits(nsplit, SimpleNamespace(host=[(b, 1, 700, b) for b in range(B)]), heads)
        assert 1 <= n <= H.LATENT_SPLITS[nsplit] and n & n - 1 == 0
        assert n == 1 or n * B * groups <= 256
        assert n == H.LATENT_SPLITS[nsplit] or 2 * n * B * groups > 256
    mixed = SimpleNamespace(host=[(0, 1, 100_000, 0)] + [(b, 1, 20, b) for b in range(1, 64)])
    assert H.latent_splits(nsplit, mixed, heads) == min(H.LATENT_SPLITS[nsplit], 128 // (1 << (groups - 1).bit_length()))
