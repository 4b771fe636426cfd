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
    """A captured launch keeps counters of its own: replays while eager launches of the same
    product run on another stream give the eager result, every time, and so do those."""
    from cake_amd.ops import gemm as G
    x = torch.randn(500, 4096, device="cuda").to(torch.bfloat16)
    w = (torch.randn(4096, 4096, device="cuda") * 2.0 ** -6).to(torch.bfloat16)
    want = G.linear(x, w, cfg=27, splits=2)
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    held = [torch.empty_like(want) for _ in range(4)]
    outs = [[torch.zeros_like(want) for _ in range(12)] for _ in range(2)]
    with torch.cuda.stream(side):
        G.linear(x, w, cfg=27, splits=2)   # its workspace and counters
    with torch.cuda.graph(graph):
        for o in held:
            G.linear(x, w, cfg=27, splits=2, out=o)
    torch.cuda.synchronize()
    for i in range(3):   # nothing waits between the two streams
        graph.replay()
        for o, h in zip(outs[0][4 * i:], held):
            o.copy_(h)
        with torch.cuda.stream(side):
            for o in outs[1][4 * i:4 * i + 4]:
                G.linear(x, w, cfg=27, splits=2, out=o)
    torch.cuda.synchronize()
    assert all(torch.equal(o, want) for side_outs in outs for o in side_outs)


def test_graphs_side_by_side_keep_their_slabs(cuda):
    """Two graphs, captured one after the other and replayed on two streams at once: pieces of a
    tile (cfg 27) and slabs with a second launch (cfg 0), the eager result every time."""
    from cake_amd.ops import gemm as G
    x = torch.randn(2, 500, 4096, device="cuda").to(torch.bfloat16)
    w = (torch.randn(4096, 4096, device="cuda") * 2.0 ** -6).to(torch.bfloat16)
    plans = [(27, 2), (0, 2)] * 3
    want = [[G.linear(x[g], w, cfg=c, splits=s) for c, s in plans] for g in range(2)]
    outs = [[torch.zeros_like(o) for o in row] for row in want]
    graphs, streams = [torch.cuda.CUDAGraph() for _ in range(2)], [torch.cuda.Stream() for _ in range(2)]
    for g, graph in enumerate(graphs):
        with torch.cuda.graph(graph):
            for (c, s), o in zip(plans, outs[g]):
                G.linear(x[g], w, cfg=c, splits=s, out=o)
    torch.cuda.synchronize()
    for _ in range(3):
        for _ in range(4):
            for graph, st in zip(graphs, streams):
                with torch.cuda.stream(st):
                    graph.replay()
        torch.cuda.synchronize()
        for g in range(2):
            assert all(torch.equal(o, e) for o, e in zip(outs[g], want[g]))
            for o in outs[g]:
                o.zero_()
        torch.cuda.synchronize()


def test_counters_are_of_a_stream_or_of_a_capture(cuda, monkeypatch):
    """Launches that may run side by side never share counters, however many there were; a stream's
    stay its own and zero; the newest 16 streams keep theirs."""
    from cake_amd.ops import gemm as G
    monkeypatch.setattr(G, "_ticks", {})
    dev = torch.empty(1, device="cuda").device

    def here():
        return G._counters(dev, torch.cuda.current_stream().cuda_stream)
    streams = [torch.cuda.Stream() for _ in range(20)]
    mine = here()
    eager = []
    for s in streams[:15]:
        with torch.cuda.stream(s):
            eager.append(here())
    for _ in range(5000):
        assert here() is mine
    for s, t in zip(streams, eager):
        with torch.cuda.stream(s):
            assert here() is t
    captured, graphs = [], [torch.cuda.CUDAGraph() for _ in range(3)]
    for g in graphs:   # one after the other on PyTorch's one capture stream
        with torch.cuda.graph(g):
            captured.append(here())
            assert here() is captured[-1]
    ptrs = {t.data_ptr() for t in [mine, *eager, *captured]}
    assert len(ptrs) == 1 + len(eager) + len(captured)
    for s in streams:   # more streams than are kept
        with torch.cuda.stream(s):
            assert not bool(here().any())
    assert len(G._ticks) <= 16 and here() is not mine and not bool(here().any())
    captured[0].fill_(7)   # another use of the graph's pool: a replay starts from zero
    graphs[0].replay()
    torch.cuda.synchronize()
    assert not bool(captured[0].any())


def test_many_captures_keep_their_pieces(cuda):
    """The thousandth capture runs the same kernel as the first: the same bits."""
    from cake_amd.ops import gemm as G
    x = torch.randn(130, 512, device="cuda").to(torch.bfloat16)
    w = torch.randn(256, 512, device="cuda").to(torch.bfloat16)

    def product(out, splits=3):
        return G.linear(x, w, epi="store32", resid=out, cfg=27, splits=splits)
    want = product(torch.empty(130, 256, device="cuda"))
    assert not torch.equal(want, product(torch.empty_like(want), 1))   # sums in another order
    for _ in range(5):
        graph, outs = torch.cuda.CUDAGraph(), [torch.empty_like(want) for _ in range(500)]
        with torch.cuda.graph(graph):
            for o in outs:
                product(o)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(o, want) for o in outs)


def test_a_graph_holds_the_counters_of_pieces(cuda):
    """A captured product's counters are as many as tiles in pieces have, not the stream form's, which every replay would
    clear too; pieces of the most tiles find them zero and leave them so."""
    from cake_amd.ops import gemm as G
    M, N, K = 4096, 4096, 1024
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = torch.randn(N, K, device="cuda").bfloat16() * K ** -0.5
    G._graph_ticks.clear()
    outs = []
    for cfg, splits in ((22, 1), (35, 3)):
        want = G.linear(x, w, epi="store32", resid=torch.empty(M, N, device="cuda"), cfg=cfg, splits=splits)
        graph, out = torch.cuda.CUDAGraph(), torch.zeros(M, N, device="cuda")
        with torch.cuda.graph(graph):
            G.linear(x, w, epi="store32", resid=out, cfg=cfg, splits=splits)
        outs.append((graph, out, want))
    (_, ticks), = G._graph_ticks.values()
    assert ticks.numel() == G._lib().cake_gemm_ticks() < G._lib().cake_gemm_rows_ticks()
    for _ in range(3):
        for graph, out, want in outs:
            out.zero_()
            graph.replay()
            assert torch.equal(out, want)
    assert not bool(ticks.any())
