"""Four-wave tiles of every height and width (gemm_4w.h): edges, short k, pieces, gated pairs."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# one k step up to more than a buffer holds; rows and columns one off the tile's edge; in pieces
@pytest.mark.parametrize("cfg", range(27, 39))
@pytest.mark.parametrize("rows,cols,K,splits", [(-1, 1, 64, 1), (1, -3, 192, 1), (0, 0, 320, 1), (3, 5, 1088, 4)])
@pytest.mark.parametrize("epi", ["store", "resid32", "swiglu"])
def test_tile_edges(cuda, cfg, rows, cols, K, splits, epi):
    """f32 sums of 16-bit products, in two orders, one rounding to bf16 (of gate, up and result in the
    gated form); the same bits every time."""
    from cake_amd.ops import gemm as G
    bm, bn = G.CFG_TILES[cfg]
    M, N = 2 * bm + rows, 3 * bn + cols
    if epi == "swiglu":
        N = 2 * (N // 32 * 16)
    g = torch.Generator(device="cuda").manual_seed(cfg + K)
    x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).to(torch.bfloat16)
    y = x.float() @ w.float().t()
    if epi == "swiglu":
        y = torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:]
    outs = []
    for _ in range(2):
        r = torch.zeros(M, N, device="cuda") if epi == "resid32" else None
        outs.append(G.linear(x, w, epi=epi, resid=r, cfg=cfg, splits=splits))
    assert torch.equal(outs[0], outs[1])
    tol = K * 2.0 ** -21 + (2.0 ** -16 if epi == "resid32" else 2.0 ** -8)
    scale = y.pow(2).mean().sqrt() + y.abs()
    assert bool(((outs[0].float() - y).abs() <= tol * scale).all())


# the other type and the other epilogues that plans take: whole tiles and pieces, ragged edges
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("cfg", range(27, 39))
@pytest.mark.parametrize("K,splits", [(192, 1), (1088, 4)])
@pytest.mark.parametrize("epi", ["store", "swiglu", "store32", "silu", "quick_gelu", "gelu", "relu2"])
def test_types_and_epilogues(cuda, dt, cfg, K, splits, epi):
    """f32 sums within K 2^-22 of the exact ones' scale (an activation's slope is at most 1.2, relu2's 2 |y|)
    and one rounding to the type: 2^-8 (bf16) or 2^-11; activations of their own 2^-10."""
    from cake_amd.ops import gemm as G
    bm, bn = G.CFG_TILES[cfg]
    M, N = bm + 33, bn + 24
    if epi == "swiglu":
        N = 2 * (N // 32 * 16)
    g = torch.Generator(device="cuda").manual_seed(cfg + K)
    x = torch.randn(M, K, device="cuda", generator=g).to(dt)
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).to(dt)
    y = x.double() @ w.double().t()
    f = torch.nn.functional
    want = {"swiglu": lambda: f.silu(y[:, :N // 2]) * y[:, N // 2:], "silu": lambda: f.silu(y),
            "quick_gelu": lambda: y * torch.sigmoid(1.702 * y), "gelu": lambda: f.gelu(y),
            "relu2": lambda: torch.relu(y).square()}.get(epi, lambda: y)()
    r = torch.zeros(M, N, device="cuda") if epi == "store32" else None
    got = G.linear(x, w, epi=epi, resid=r, cfg=cfg, splits=splits)
    size = 2.0 ** -16 if epi == "store32" else 2.0 ** (-8 if dt == torch.bfloat16 else -11)
    own = 0. if epi in ("store", "store32") else 2.0 ** -10
    sums = K * 2.0 ** -22 * (1 + y.abs().max().item()) * 2
    assert bool(((got.double() - want).abs() <= (size + own) * want.abs() + sums).all())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("cfg", range(28, 39))
@pytest.mark.parametrize("epi", ["add16", "geglu"])
def test_image_epilogues_run_on_another_tile(cuda, dt, cfg, epi):
    """Tiles without these epilogues: the call's result is the 128 x 256 tile's, pieces or none."""
    from cake_amd.ops import gemm as G
    M, N, K = 300, 288, 1088
    g = torch.Generator(device="cuda").manual_seed(cfg)
    x = torch.randn(M, K, device="cuda", generator=g).to(dt)
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).to(dt)
    kw = {"resid": torch.randn(M, N, device="cuda", generator=g).to(dt)} if epi == "add16" else {}
    want = G.linear(x, w, epi=epi, cfg=27, splits=1, **kw)
    assert all(torch.equal(G.linear(x, w, epi=epi, cfg=cfg, splits=s, **kw), want) for s in (1, 4))
