"""Grouped products by tile heights (gemm_inst_grouped.hip): rows of up to 1024 columns, on the four-wave tiles of gemm_4w.h,
and some of more, on those of gemm_ws.h (which have their own tests too)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg", [0, 1, 2])
@pytest.mark.parametrize("N,K,ld", [(8, 8, 8), (257, 128, 136), (300, 200, 200), (520, 1096, 1104), (40, 72, 1 << 22)])
def test_tile_heights(cuda, cfg, N, K, ld):
    """Groups of none, of a tile and one row to either side, rows far apart: one rounding to bf16
    (2^-8) of f32 sums; nothing beside the rows is written."""
    from cake_amd.ops import gemm as G
    bm = G.GROUPED_CFGS[cfg]
    counts = [bm - 1, 0, bm, bm + 1, 1, 2 * bm + 33]
    R = sum(counts)
    g = torch.Generator(device="cuda").manual_seed(N)
    x = torch.empty((R - 1) * ld + K, dtype=torch.bfloat16, device="cuda").as_strided((R, K), (ld, 1))
    x.copy_(torch.randn(R, K, device="cuda", generator=g))
    w = (torch.randn(len(counts), N, K, device="cuda", generator=g) * K ** -0.5).to(torch.bfloat16)
    tiles, r0, want = [], 0, []
    for e, c in enumerate(counts):
        tiles += [[e, r0 + t, min(bm, c - t), 0] for t in range(0, c, bm)]
        want.append(x[r0:r0 + c].float() @ w[e].float().t())
        r0 += c
    t = torch.tensor(tiles + [[0, 0, 0, 0], [len(tiles), 0, 0, 0]], dtype=torch.int32, device="cuda")
    out = torch.full((R, N + 8), 7.0, dtype=torch.bfloat16, device="cuda")
    G.grouped(x, w, t, cfg, out[:, :N])
    want = torch.cat(want)
    assert bool((out[:, N:] == 7.0).all())
    assert bool(((out[:, :N].float() - want).abs() <= 2.0 ** -8 * want.abs() + K * 2.0 ** -20).all())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("cfg", [0, 1, 2, 5, 6])
@pytest.mark.parametrize("epi", ["silu", "relu2"])
def test_activations_of_every_height(cuda, dt, cfg, epi):
    """Short rows, the four-wave tiles: 16-bit types and activations; configuration 6 by the list's height.  One
    rounding (2^-8, 2^-11) of f32 sums, the activation's own 2^-10."""
    from cake_amd.ops import gemm as G
    N, K = 300, 200
    for bm in ((128, 160, 192, 256) if cfg == 6 else (G.GROUPED_CFGS[cfg],)):
        counts = [bm + 1, 3, 0, bm, bm - 1]
        R = sum(counts)
        g = torch.Generator(device="cuda").manual_seed(bm)
        x = torch.randn(R, K, device="cuda", generator=g).to(dt)
        w = (torch.randn(len(counts), N, K, device="cuda", generator=g) * K ** -0.5).to(dt)
        tiles, r0, y = [], 0, []
        for e, c in enumerate(counts):
            tiles += [[e, r0 + t, min(bm, c - t), 0] for t in range(0, c, bm)]
            y.append(x[r0:r0 + c].double() @ w[e].double().t())
            r0 += c
        t = torch.tensor(tiles + [[0, 0, 0, 0], [len(tiles), bm, 0, 0]], dtype=torch.int32, device="cuda")
        out = torch.full((R, N + 8), 7.0, dtype=dt, device="cuda")
        G.grouped(x, w, t, cfg, out[:, :N], epi=epi)
        y = torch.cat(y)
        want = torch.nn.functional.silu(y) if epi == "silu" else torch.relu(y).square()
        size = 2.0 ** (-8 if dt == torch.bfloat16 else -11) + 2.0 ** -10
        assert bool((out[:, N:] == 7.0).all())
        assert bool(((out[:, :N].double() - want).abs() <= size * want.abs() + K * 2.0 ** -22 * (1 + y.abs()) * 2).all())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=str)
def test_a_k_of_their_own(cuda, dt):
    """Weight rows of 4 KB and 256 tiles and more: every tile starts at another k and goes round.  One rounding
    (2^-8, 2^-11) of f32 sums."""
    from cake_amd.ops import gemm as G
    N, K, bm = 520, 2048, 256
    counts = [(7 * e) % 41 + (200 if e % 31 == 0 else 0) for e in range(90)]
    R = sum(counts)
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(R, K, device="cuda", generator=g).to(dt)
    w = (torch.randn(len(counts), N, K, device="cuda", generator=g) * K ** -0.5).to(dt)
    tiles, r0, y = [], 0, []
    for e, c in enumerate(counts):
        tiles += [[e, r0 + t, min(bm, c - t), 0] for t in range(0, c, bm)]
        y.append(x[r0:r0 + c].double() @ w[e].double().t())
        r0 += c
    assert len(tiles) * 3 >= 256
    t = torch.tensor(tiles + [[0, 0, 0, 0], [len(tiles), bm, 0, 0]], dtype=torch.int32, device="cuda")
    out = torch.full((R, N + 8), 7.0, dtype=dt, device="cuda")
    G.grouped(x, w, t, 6, out[:, :N])
    y = torch.cat(y)
    size = 2.0 ** (-8 if dt == torch.bfloat16 else -11)
    assert bool((out[:, N:] == 7.0).all())
    assert bool(((out[:, :N].double() - y).abs() <= size * y.abs() + K * 2.0 ** -22 * (1 + y.abs())).all())
