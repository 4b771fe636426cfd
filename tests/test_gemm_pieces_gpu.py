"""Four-wave tiles in k pieces (gemm_4w.h): the piece sums, their order, their counters."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# 64 / 30 / 12 tiles; 258 = one wave + 2 tiles; k steps that the pieces divide and do not
@pytest.mark.parametrize("cfg,M,N,K,splits", [
    (22, 777, 4096, 1024, 4), (25, 300, 3840, 1856, 8), (23, 300, 1000, 2624, 16),
    (26, 11000, 1152, 704, 3), (24, 129, 1500, 4096, 5), (27, 2000, 4000, 640, 2)])
@pytest.mark.parametrize("epi", ["store", "resid32", "gelu"])
def test_pieces_sum_to_the_product(cuda, cfg, M, N, K, splits, epi):
    """f32 sums of 16-bit products: within K 2^-22 of the row's scale before the result is rounded
    (bf16, 2^-8 of it), the same bits every time, and a second launch finds clean counters."""
    from cake_amd.ops import gemm as G
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).to(torch.bfloat16)
    want = x.float() @ w.float().t()
    if epi == "gelu":
        want = torch.nn.functional.gelu(want)
    outs = []
    for _ in range(3):
        r = torch.zeros(M, N, device="cuda") if epi == "resid32" else None
        outs.append(G.linear(x, w, epi=epi, resid=r, cfg=cfg, splits=splits))
    assert all(torch.equal(o, outs[0]) for o in outs[1:])
    # two f32 sums in different orders, one rounding to bf16, GELU's own 2^-20
    tol = K * 2.0 ** -21 + (2.0 ** -16 if epi == "resid32" else 2.0 ** -8)
    scale = want.pow(2).mean().sqrt() + want.abs()
    assert bool(((outs[0].float() - want).abs() <= tol * scale).all())


def test_pieces_in_a_graph_beside_eager_work(cuda):
    """A captured launch keeps counters of its own: replays beside eager launches of the same
    product on another stream give the eager result, every time."""
    from cake_amd.ops import gemm as G
    x = torch.randn(500, 4096, device="cuda").to(torch.bfloat16)
    w = (torch.randn(4096, 4096, device="cuda") * 2.0 ** -6).to(torch.bfloat16)
    want = G.linear(x, w, cfg=27, splits=2)
    out = torch.empty_like(want)
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    G._workspace(x.device, 1 << 26)
    with torch.cuda.graph(graph):
        G.linear(x, w, cfg=27, splits=2, out=out)
    for _ in range(4):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        with torch.cuda.stream(side):
            assert torch.equal(G.linear(x, w, cfg=27, splits=2), want)
        torch.cuda.synchronize()
