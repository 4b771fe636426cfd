"""Grouped products on the four-wave tiles: groups around a tile's rows, columns and k around its
edges, rows too far apart for the tiles' 32-bit offsets."""
import pytest
import torch

from cake_amd.ops import gemm as G

pytestmark = pytest.mark.gpu

# one rounding of the result: half a unit in the last place (sums are float32, K 2^-24 below it)
TOL = {torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11}


def _tiles(counts, bm):
    tiles, r0 = [], 0
    for e, c in enumerate(counts):
        tiles += [[e, r0 + t, min(bm, c - t), 0] for t in range(0, c, bm)]
        r0 += c
    return tiles


def _check(x, w, counts, cfg, dt, out):
    R, (E, N, K) = x.shape[0], w.shape
    tiles = _tiles(counts, G.GROUPED_CFGS[cfg])
    t = torch.tensor(tiles + [[0, 0, 0, 0], [len(tiles), 0, 0, 0]], dtype=torch.int32, device="cuda")
    G.grouped(x, w, t, cfg, out)
    r0 = 0
    for e, c in enumerate(counts):
        want = x[r0:r0 + c].cpu().double() @ w[e].cpu().double().t()
        got = out[r0:r0 + c].cpu().double()
        assert c == 0 or float((got - want).norm() / want.norm()) < TOL[dt], (e, c)
        r0 += c
    assert r0 == R


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("cfg", [0, 5])
@pytest.mark.parametrize("N,K", [(8, 8), (255, 64), (256, 72), (257, 128), (520, 184), (100, 1000)])
def test_edges(dt, cfg, N, K):
    bm = G.GROUPED_CFGS[cfg]
    counts = [bm - 1, 0, bm, bm + 1, 1, 2 * bm + bm // 2 + 1, 33]
    g = torch.Generator().manual_seed(N + K)
    x = torch.randn(sum(counts), K + 8, generator=g).to(dt).cuda()[:, :K]
    # a neighbour's values must not come in through a row's tail
    w = (torch.randn(len(counts), N, K, generator=g) * K ** -0.5).to(dt).cuda()
    buf = torch.full((sum(counts), N + 8), 7.0, dtype=dt, device="cuda")
    _check(x, w, counts, cfg, dt, buf[:, :N])
    assert bool((buf[:, N:] == 7.0).all())


@pytest.mark.parametrize("cfg", [0, 5])
def test_far_rows(cfg):
    dt, K, ld = torch.bfloat16, 72, 1 << 22
    counts = [3, G.GROUPED_CFGS[cfg] + 70]
    R = sum(counts)
    x = torch.empty((R - 1) * ld + K, dtype=dt, device="cuda").as_strided((R, K), (ld, 1))
    x.copy_(torch.randn(R, K).to(dt))
    w = (torch.randn(2, 40, K) * K ** -0.5).to(dt).cuda()
    _check(x, w, counts, cfg, dt, torch.empty(R, 40, dtype=dt, device="cuda"))
