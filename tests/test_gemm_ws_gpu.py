"""Tiles whose operands are asked for by waves of their own (gemm_ws.h): groups of routed rows, f32 results."""
import pytest
import torch

pytestmark = pytest.mark.gpu
SIZE = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _tiles(counts, bm):
    out, r0 = [], 0
    for e, c in enumerate(counts):
        out += [[e, r0 + t, min(bm, c - t), 0] for t in range(0, c, bm)]
        r0 += c
    return out


def _groups(cuda, dt, cfg, counts, N, K, bm, lda=0):
    """Rows of every group against f32 sums (two orders: K 2^-21 of the scale) rounded once; nothing beside
    them is written, and a second launch gives the same bits."""
    from cake_amd.ops import gemm as G
    R, E = sum(counts), len(counts)
    lda = lda or K
    g = torch.Generator(device="cuda").manual_seed(R + N)
    x = torch.empty((R - 1) * lda + K, dtype=dt, device="cuda").as_strided((R, K), (lda, 1))
    x.copy_(torch.randn(R, K, device="cuda", generator=g))
    w = torch.empty(E, N, K, dtype=dt, device="cuda").normal_(0, K ** -0.5, generator=g)
    tiles = _tiles(counts, bm)
    t = torch.tensor(tiles + [[0, 0, 0, 0], [len(tiles), bm, 0, 0]], dtype=torch.int32, device="cuda")
    out = torch.full((R, N + 8), 7.0, dtype=dt, device="cuda")
    again = torch.empty_like(out)
    G.grouped(x, w, t, cfg, out[:, :N])
    G.grouped(x, w, t, cfg, again[:, :N])
    assert bool((out[:, N:] == 7.0).all()) and torch.equal(out[:, :N], again[:, :N])
    r0 = 0
    for e, c in enumerate(counts):
        want = x[r0:r0 + c].float() @ w[e].float().t()
        tol = SIZE[dt] * want.abs() + K * 2.0 ** -21 * (1 + want.abs())
        assert bool(((out[r0:r0 + c, :N].float() - want).abs() <= tol).all()), (e, c)
        r0 += c


# every height, by configuration and by the list; few tiles (128 columns) and many; a k that ends amid a step, rows
# farther apart than they are long; groups of none, of one row, of a tile and one row to either side
@pytest.mark.parametrize("dt", list(SIZE), ids=str)
@pytest.mark.parametrize("cfg,bm", [(0, 128), (1, 160), (2, 192), (3, 224), (5, 256), (6, 160), (6, 192), (6, 224), (6, 256)])
@pytest.mark.parametrize("N,K", [(8, 1032), (300, 1096), (3000, 1152)])
def test_groups_of_every_height(cuda, dt, cfg, bm, N, K):
    counts = [bm - 1, 0, bm, bm + 1, 1, 2 * bm + 33, 16, 17]
    _groups(cuda, dt, cfg, counts, N, K, bm, K + 8)


@pytest.mark.parametrize("bm", [160, 192, 224, 256])
def test_more_tiles_than_workgroups_on_cold_weights(cuda, bm):
    """Several tiles a workgroup, one after the other, whose weights no cache holds (0.5 GB): all that a step
    reads has landed."""
    _groups(cuda, torch.bfloat16, 6, [bm - (7 * e) % 60 for e in range(48)], 2600, 2048, bm)


def test_groups_of_several_tiles(cuda):
    """Tiles that share their weights and tiles that read them alone, side by side."""
    _groups(cuda, torch.float16, 6, [700, 3, 160, 480, 161, 0, 90, 1000], 2048, 1536, 160)


def _height(counts, F, W):
    """(cost, height) of every height, in 64 bits."""
    R, out = sum(counts), []
    mem = (len(counts) * F * W + R * (F + W)) * 2 / 5.8e6

    def us(q, t, n, k):
        few = t * -(-n // 256) <= (128 if q == 0 else 64)
        body = 3 if few and q else q
        whole, part = divmod(t * -(-n // (128 if few else 256)) / 256, 1)
        rounds = whole + (min(1.0, 0.82 + 1.42 * part) if part else 0.0)
        step, end = (1.124, 1.152, 1.299, 1.339)[body], (5.53, 7.80, 7.07, 8.42)[body]
        return max(rounds * (step * (0.448 if few else 1) * -(-k // 64) + end * (1.54 if few else 1)), mem)
    for q, bm in enumerate((160, 192, 224, 256)):
        t = sum(-(-c // bm) for c in counts)
        out.append((us(q, t, F, W) + us(q, t, W, F), bm))
    return out


@pytest.mark.parametrize("counts,F,W", [([64], 72, 1032), ([161, 160, 159, 1], 300, 1160), ([192, 193, 191] * 20, 1096, 1100),
                                        ([220] * 64, 520, 2048), ([225, 224, 0, 223, 500] * 9, 1500, 1032),
                                        ([250] * 40 + [1] * 30, 2000, 1536), ([150] * 64, 1856, 2048)])
def test_height_of_the_groups(cuda, counts, F, W):
    """The device lists tiles of the cheapest height (of two within 1e-4 either), every row in one of them."""
    from cake_amd.ops import experts as X
    from cake_amd.ops import gemm as G
    E, R = len(counts), sum(counts)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    ids = ids[torch.randperm(R, generator=torch.Generator().manual_seed(1))].int().cuda().view(R, 1)
    p = X.plan(ids, torch.ones(R, 1, device="cuda"), E, torch.bfloat16, F * W, F)
    assert p.cfg == G.BY_LIST
    n, bm = p.tiles[-1, :2].tolist()
    costs = _height(counts, F, W)
    assert bm in [b for c, b in costs if c <= min(costs)[0] * (1 + 1e-4)]
    assert p.tiles[:n].tolist() == _tiles(counts, bm)


# f32 results: fewer tiles than workgroups and more, pieces alone and behind whole tiles, bias and factor
@pytest.mark.parametrize("dt", list(SIZE), ids=str)
@pytest.mark.parametrize("cfg", [22, 25, 34, 35])
@pytest.mark.parametrize("M,N,K,splits", [(1, 8, 64, 1), (700, 1000, 448, 3), (1500, 12300, 192, 1), (2100, 8200, 512, 2)])
@pytest.mark.parametrize("epi", ["resid32", "store32"])
def test_f32_results(cuda, dt, cfg, M, N, K, splits, epi):
    """f32 sums of 16-bit products in two orders: K 2^-21 of the scale, twice that with the factor; the same bits
    every time, and a second launch finds clean counters."""
    from cake_amd.ops import gemm as G
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, device="cuda", generator=g).to(dt)
    w = torch.empty(N, K, device="cuda", dtype=dt).normal_(0, K ** -0.5, generator=g)
    bias = torch.randn(N, device="cuda", generator=g).to(dt)
    y = 0.5 * (x.float() @ w.float().t() + bias.float())
    outs = []
    for _ in range(3):
        r = torch.full((M, N + 4), 3.0, device="cuda")
        G.linear(x, w, bias, epi=epi, resid=r[:, :N], alpha=0.5, cfg=cfg, splits=splits)
        assert bool((r[:, N:] == 3.0).all())
        outs.append(r)
    assert all(torch.equal(o, outs[0]) for o in outs[1:])
    want = y + 3.0 if epi == "resid32" else y
    assert bool(((outs[0][:, :N] - want).abs() <= K * 2.0 ** -20 + 2.0 ** -21 * want.abs()).all())
