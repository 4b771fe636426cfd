"""Splits of latent decode by the sequences of a step."""
from types import SimpleNamespace

import pytest
import torch

from cake_amd.models.hybrid import model as H
from cake_amd.ops import latent as LA


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
    mixed = SimpleNamespace(host=[(0, 1, 10_000, 0)] + [(b, 1, 20, b) for b in range(1, 64)])
    assert H.latent_splits(nsplit, mixed, heads) == min(H.LATENT_SPLITS[nsplit], 128 // (1 << (groups - 1).bit_length()))
    # short sequences of up to a tenth of its keys count nothing
    mixed = SimpleNamespace(host=[(0, 1, 100_000, 0)] + [(b, 1, 20, b) for b in range(1, 64)])
    assert H.latent_splits(nsplit, mixed, heads) == min(H.LATENT_SPLITS[nsplit], 256 // (1 << (groups - 1).bit_length()))
    # more where a CU holds two workgroups, as long as a split has four tiles
    for B, keys in ((1, 700), (3, 3000), (24, 3000), (3, 30_000), (300, 30_000)):
        rows = SimpleNamespace(host=[(b, 1, keys - 1, b) for b in range(B)])
        one, two = (H.latent_splits(nsplit, rows, heads, p) for p in (1, 2))
        assert two in (one, 2 * one) and (two == one or two * B * groups <= 512 and keys > 192 * two)
        assert two > one or 2 * one > H.LATENT_SPLITS[nsplit] or 2 * one * B * groups > 512 or keys <= 384 * one


@pytest.mark.parametrize("rank,heads,dtype,per_cu,short", [(512, 16, torch.bfloat16, 1, True), (512, 128, torch.bfloat16, 1, False),
                                                           (256, 128, torch.float16, 2, True), (1024, 32, torch.bfloat16, 1, True),
                                                           (256, 16, torch.float32, 2, True), (512, 16, torch.float32, 1, True)])
def test_workgroups_of_a_cu_and_tiles_alone(rank, heads, dtype, per_cu, short):
    """As the kernel's LDS has it; 32-key tiles in short contexts while a sequence's sums are few."""
    sh = LA.LatentShape(heads=heads, dim=128, rot_dim=64, vdim=128, q_rank=1536, kv_rank=rank, rot_pairs=32)
    assert LA.decode_per_cu(sh, dtype) == per_cu
    assert H.latent_alone(1, sh) == ((8, 32) if short else (4, 64)) and H.latent_alone(8, sh) == (16, 64)
