"""Latent decode in 32-key tiles: the same attention as in 64-key ones."""
import pytest
import torch

from cake_amd.ops import latent as LA

pytestmark = pytest.mark.gpu


# one key, a tile and one to either side, a split's end, all of the cache; more splits than tiles and fewer
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32], ids=str)
@pytest.mark.parametrize("rank,heads", [(512, 32), (200, 5), (1024, 16)])
@pytest.mark.parametrize("nsplit", [1, 3, 8, 64])
def test_tile_of_32(cuda, dt, rank, heads, nsplit):
    """Value sums of the same keys against 64 bits: the weights p are rounded to the storage type as in 64-key tiles, so
    the error of either, relative to the largest value, stays under a step of it."""
    sh = LA.LatentShape(heads=heads, dim=64, rot_dim=32, vdim=24, q_rank=64, kv_rank=rank, rot_pairs=16)
    S, lens = 256, [1, 31, 32, 33, 64, 97, 255, 256]
    B = len(lens)
    g = torch.Generator(device="cuda").manual_seed(rank + nsplit)
    cache = torch.randn(B, S, sh.LD, device="cuda", generator=g).to(dt)
    for b, n in enumerate(lens):
        cache[b, n:] = float("nan")
    qa = (torch.randn(B, heads, sh.LD, device="cuda", generator=g) * 0.3).to(dt)
    uv = torch.randn(heads, sh.DVP, sh.RP, device="cuda", generator=g).to(dt)
    pos = torch.tensor(lens, dtype=torch.int32, device="cuda") - 1
    slot = torch.arange(B, dtype=torch.int32, device="cuda")
    clean = torch.nan_to_num(cache)
    step = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -18}[dt]
    for tile in (32, 64):
        part = torch.full((sh.part_floats(B, nsplit),), float("nan"), device="cuda")
        y = torch.empty(B, heads * 24, device="cuda", dtype=dt)
        LA.decode(sh, qa, pos, slot, clean, 0.05, nsplit, part, tile)
        LA.out(sh, part, pos, uv, nsplit, y, tile)
        for b, n in enumerate(lens):
            k = cache[b, :n].double()
            p = torch.softmax(0.05 * qa[b].double() @ k.t(), -1)
            want = torch.einsum("hvr,hr->hv", uv[:, :24].double().cpu(), (p @ k[:, :sh.RP]).cpu()).flatten()
            assert (y[b].double().cpu() - want).abs().max() <= 3 * step * want.abs().max(), (tile, n)
    with pytest.raises(RuntimeError):
        LA.decode(sh, qa, pos, slot, clean, 0.05, nsplit, part, 16)
