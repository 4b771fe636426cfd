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


@pytest.mark.parametrize("dt", list(SIZE), ids=str)
@pytest.mark.parametrize("bm", [160, 192, 224, 256])
@pytest.mark.parametrize("E", [2, 9], ids=["few", "many"])
@pytest.mark.parametrize("epi", ["silu", "quick_gelu", "gelu", "relu2"])
def test_activations(cuda, dt, bm, E, epi):
    """As routed experts run them, on narrow tiles of few and on all of many: one rounding (2^-8, 2^-11) of f32 sums, the
    activation's own 2^-10 and its factor of at most 2 on what the sums differ by."""
    from cake_amd.ops import gemm as G
    N, K = 2600, 1096
    counts = [bm, bm - 1, bm + 1, 0, 3, 2 * bm, 17, 5 * bm, bm][:E]
    R = sum(counts)
    g = torch.Generator(device="cuda").manual_seed(bm)
    x = torch.randn(R, K, device="cuda", generator=g).to(dt)
    w = torch.empty(E, N, K, dtype=dt, device="cuda").normal_(0, K ** -0.5, generator=g)
    tiles = _tiles(counts, bm)
    t = torch.tensor(tiles + [[0, 0, 0, 0], [len(tiles), bm, 0, 0]], dtype=torch.int32, device="cuda")
    out = torch.full((R, N + 8), 7.0, dtype=dt, device="cuda")
    G.grouped(x, w, t, 6, out[:, :N], epi=epi)
    F = torch.nn.functional
    act = {"silu": F.silu, "gelu": F.gelu, "quick_gelu": lambda y: y * torch.sigmoid(1.702 * y), "relu2": lambda y: F.relu(y).square()}[epi]
    y = torch.cat([x[r:r + c].float() @ w[e].float().t() for e, (r, c) in enumerate(zip([sum(counts[:e]) for e in range(E)], counts))])
    want = act(y.double())
    tol = (SIZE[dt] + 2.0 ** -10) * want.abs() + 2 * K * 2.0 ** -21 * (1 + y.abs())
    assert bool((out[:, N:] == 7.0).all()) and bool(((out[:, :N].double() - want).abs() <= tol).all())


@pytest.mark.parametrize("bm", [160, 192, 224, 256])
def test_more_tiles_than_workgroups_on_cold_weights(cuda, bm):
    """Several tiles a workgroup, one after the other, whose weights no cache holds (0.5 GB): all that a step
    reads has landed."""
    _groups(cuda, torch.bfloat16, 6, [bm - (7 * e) % 60 for e in range(48)], 2600, 2048, bm)


def test_groups_of_several_tiles(cuda):
    """Tiles that share their weights and tiles that read them alone, side by side."""
    _groups(cuda, torch.float16, 6, [700, 3, 160, 480, 161, 0, 90, 1000], 2048, 1536, 160)


def _height(counts, F, W):
    """(cost, height) of every height, in 64 bits: each product as on the tiles that its own k takes."""
    R, out = sum(counts), []
    size = (len(counts) * F * W + R * (F + W)) * 2

    def us(bm, t, n, k):
        if k <= 1024:
            step, end = {128: (1.106, 5.4), 160: (1.161, 7.76), 192: (1.38, 8.64), 224: (1.422, 9.39), 256: (1.547, 11.64)}[bm]
            return max(-(-t * -(-n // 256) // 256) * (step * -(-k // 64) + end), size / 8.2e6)
        q = max(bm // 32 - 5, 0)
        few = t * -(-n // 256) <= (128 if q == 0 else 64)
        body = 3 if few and q else q
        r = t * -(-n // (128 if few else 256)) / 256
        whole, part = divmod(r, 1)
        rounds = whole + (min(1.0, 0.82 + 1.42 * part) if part else 0.0)
        step, end = (1.124, 1.152, 1.299, 1.339)[body], (5.53, 7.80, 7.07, 8.42)[body]
        one = step * (0.448 if few else 1) * -(-k // 64) + end * (1.54 if few else 1)
        return max(rounds * one, size / 5.8e6 + (0.5 * (rounds - r) * one if whole else 0))
    for bm in (160, 192, 224, 256) if W > 1024 else (128, 160, 192, 256):
        t = sum(-(-c // bm) for c in counts)
        out.append((us(bm, t, F, W) + us(bm, t, W, F), bm))
    return out


@pytest.mark.parametrize("counts,F,W", [([64], 72, 1032), ([161, 160, 159, 1], 300, 1160), ([192, 193, 191] * 20, 1096, 1100),
                                        ([220] * 64, 520, 2048), ([225, 224, 0, 223, 500] * 9, 1500, 1032),
                                        ([250] * 40 + [1] * 30, 2000, 1536), ([150] * 64, 1856, 2048),
                                         # a down product on the short rows' tiles under such an up product, and the other way
                                         ([192, 206, 185, 210] * 64, 512, 4096), ([240, 251, 262, 228] * 4, 2816, 1024),
                                         ([300] * 8, 4096, 1024), ([70] * 64, 1032, 1000)])
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


# a list of 224 rows, by configuration and by itself, where no tile of that height is: 193 .. 224 rows run at 256
@pytest.mark.parametrize("dt", list(SIZE), ids=str)
@pytest.mark.parametrize("cfg", [3, 6])
@pytest.mark.parametrize("N,K", [(8, 8), (300, 520), (1100, 1024)])
def test_short_rows_in_lists_of_224(cuda, dt, cfg, N, K):
    _groups(cuda, dt, cfg, [224, 0, 223, 225, 193, 192, 160, 1, 500], N, K, 224, K + 8)


@pytest.mark.parametrize("dt", list(SIZE), ids=str)
@pytest.mark.parametrize("F,W", [(768, 1160), (1024, 1032), (1032, 1024), (1304, 520)])
def test_up_and_down_on_either_side_of_the_line(cuda, dt, F, W):
    """Both products of a plan whose k lie to either side of the short rows' line: f32 sums of two orders, rounded once."""
    from cake_amd.ops import experts as X
    counts = [161, 0, 224, 193, 225, 256, 70, 129]
    R, E = sum(counts), len(counts)
    g = torch.Generator(device="cuda").manual_seed(F)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).int().cuda().view(R, 1)
    p = X.plan(ids, torch.ones(R, 1, device="cuda"), E, dt, F * W, F)
    x = torch.randn(R, W, device="cuda", generator=g).to(dt)
    up = torch.empty(E, F, W, dtype=dt, device="cuda").normal_(0, W ** -0.5, generator=g)
    down = torch.empty(E, W, F, dtype=dt, device="cuda").normal_(0, F ** -0.5, generator=g)
    a = torch.empty(R, F, dtype=dt, device="cuda")
    y = torch.empty(R, W, dtype=dt, device="cuda")
    X.product(x, up, p, a)
    X.product(a, down, p, y)
    r0 = 0
    for e, c in enumerate(counts):
        for got, rows, w in ((a, x, up), (y, a, down)):
            want = rows[r0:r0 + c].float() @ w[e].float().t()
            tol = SIZE[dt] * want.abs() + max(F, W) * 2.0 ** -21 * (1 + want.abs())
            assert bool(((got[r0:r0 + c].float() - want).abs() <= tol).all()), e
        r0 += c


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
