"""Products of few rows (gemm_rows.h): both forms, every epilogue, at the edges of their tiles.

Bound: operands are 16-bit, products and sums f32.  |error| <= K 2^-24 sum |x w| of the f32 sums,
far below the rounding of a 16-bit result (2^-8 bf16, 2^-11 f16 of its size); the activations'
approximations stay below 2^-11.  So 16-bit results are held to one rounding step plus K 2^-22 of
the row's scale, f32 results to K 2^-22."""
import pytest
import torch

pytestmark = pytest.mark.gpu
EPIS = ("store", "resid32", "add16", "swiglu", "geglu", "store32", "silu", "gelu", "relu2")
STEP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -10}


def product(x, w, b, r, epi, alpha):
    y = x.double() @ w.double().t()
    if b is not None:
        y = y + b.double()
    F = torch.nn.functional
    if epi in ("swiglu", "geglu"):
        a, u = y.chunk(2, 1)
        return F.silu(a) * u if epi == "swiglu" else a * F.gelu(u, approximate="tanh")
    if epi in ("silu", "gelu"):
        return getattr(F, epi)(y)
    if epi == "relu2":
        return y.clamp(min=0).pow(2)
    return {"store": y, "add16": y + r.double(), "resid32": r.double() + alpha * y,
            "store32": alpha * y}[epi]


def run(G, kind, x, w, b, r, out, epi, alpha):
    """One launch of the form `kind` through the C entry, as linear() makes it."""
    import ctypes
    M, K = x.shape
    N = out.shape[1]
    st = torch.cuda.current_stream().cuda_stream
    ws, tick = G._rows_state(x.device, M, st) if kind == 2 else (None, None)
    p = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    f32 = epi in ("resid32", "store32")
    rc = G._lib().cake_gemm_rows(
        G._DT[x.dtype], G.EPI[epi], kind, p(x), x.stride(0), p(w), w.stride(0),
        None if f32 else p(out), out.stride(0), p(b), p(out) if f32 else p(r),
        out.stride(0) if f32 else (0 if r is None else r.stride(0)), p(ws), p(tick),
        p(G._zeros16(x.device)), M, N, K, ctypes.c_float(alpha), st)
    assert rc == 0
    if tick is not None:
        torch.cuda.synchronize()
        assert not bool(tick.any())   # re-armed
    return out


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("epi", EPIS)
@pytest.mark.parametrize("kind,M,N,K", [
    (1, 1, 16, 8), (1, 16, 4096, 72), (1, 17, 4128, 1000), (1, 32, 48, 2048), (1, 5, 8208, 520),
    (2, 1, 16, 8), (2, 16, 160, 4096), (2, 17, 4112, 1032), (2, 33, 272, 8200), (2, 48, 64, 64),
    (2, 49, 8208, 520), (2, 64, 1040, 2048)])
def test_rows_epilogues_and_edges(cuda, dt, epi, kind, M, N, K):
    from cake_amd.ops import gemm as G
    g = torch.Generator(device="cuda").manual_seed(M * N + K)

    def rnd(*s):
        return torch.randn(*s, device="cuda", generator=g)
    gated = epi in ("swiglu", "geglu")
    Nv = 2 * N if gated else N
    x = rnd(M, K + 8).to(dt)[:, :K]                       # a row stride of its own
    w = (rnd(Nv, K + 16) * K ** -0.5).to(dt)[:, :K]
    b = rnd(Nv).to(dt)
    f32 = epi in ("resid32", "store32")
    r = rnd(M, N + 4) if f32 else rnd(M, N + 8).to(dt)    # rows of the result have a stride too
    whole = r.clone() if f32 else torch.full((M, N + 8), 7.0, device="cuda", dtype=dt)
    out = whole[:, :N]
    alpha = 0.5 if f32 else 1.0
    want = product(x, w, b, r[:, :N], epi, alpha)
    got = run(G, kind, x, w, b, None if f32 or epi != "add16" else r[:, :N], out, epi, alpha)
    scale = want.pow(2).mean().sqrt() + want.abs()
    tol = (K * 2.0 ** -22 + (2.0 ** -16 if f32 else STEP[dt])) * scale
    assert bool(((got.double() - want).abs() <= tol).all())
    assert bool((whole[:, N:] == (r[:, N:] if f32 else 7.0)).all())   # columns past N stay


def test_rows_sums_do_not_hang_on_arrival(cuda):
    from cake_amd.ops import gemm as G
    x = torch.randn(40, 8192, device="cuda").to(torch.bfloat16)
    w = torch.randn(2048, 8192, device="cuda").to(torch.bfloat16)
    outs = [run(G, 2, x, w, None, None, torch.empty(40, 2048, device="cuda"), "store32", 1.0)
            for _ in range(4)]
    assert all(torch.equal(o, outs[0]) for o in outs[1:])


def test_rows_keep_infinities_and_nan(cuda):
    """A row that holds them does not touch the others, in either form."""
    from cake_amd.ops import gemm as G
    x = torch.randn(24, 520, device="cuda").to(torch.bfloat16)
    w = torch.randn(272, 520, device="cuda").to(torch.bfloat16)
    x[3, 100], x[20, 519], w[271, 0] = float("inf"), float("nan"), float("-inf")
    want = x.double() @ w.double().t()
    for kind in (1, 2):
        got = run(G, kind, x, w, None, None, torch.empty(24, 272, device="cuda"), "store32", 1.0)
        fine = want.isfinite()
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
        torch.testing.assert_close(got[fine].double(), want[fine], rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("M,N,K", [(5, 2048, 2048), (13, 28672, 4096), (45, 28672, 4096),
                                   (24, 12288, 4096), (64, 4096, 4096), (65, 4096, 4096)])
def test_linear_takes_the_planned_form(cuda, M, N, K):
    """linear() equals the tile kernels on either side of the rule, eager, on two streams and
    captured (a graph holds the tile kernels or the direct form: no counters)."""
    from cake_amd.ops import gemm as G
    x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).to(torch.bfloat16)
    want = G.linear(x, w, cfg=0, splits=1).float()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        there = G.linear(x, w)
    here = G.linear(x, w)
    torch.cuda.synchronize()
    g, out = torch.cuda.CUDAGraph(), torch.empty(M, N, device="cuda", dtype=torch.bfloat16)
    with torch.cuda.graph(g):
        G.linear(x, w, out=out)
    replays = []
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        replays.append(out.clone())
    for got in (here, there, *replays):
        torch.testing.assert_close(got.float(), want, rtol=2.0 ** -7, atol=2.0 ** -7)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N,K,top,E,tokens,act", [(1640, 2048, 6, 64, 13, "relu2"), (40, 72, 2, 5, 9, None),
                                                  (128, 64, 1, 1024, 30, "gelu"), (272, 520, 3, 7, 1, None),
                                                  (4160, 8, 2, 1024, 750, "silu")])   # strips past the counters
def test_grouped_rows(cuda, dt, N, K, top, E, tokens, act):
    from cake_amd.ops import experts as X
    from cake_amd.ops import gemm as G
    g = torch.Generator(device="cuda").manual_seed(N)
    logits = torch.randn(tokens, E, device="cuda", generator=g)
    p = X.plan(*X.route(logits, top), E, dt)
    assert (p.cfg == G.ROWS) == (tokens * top <= 4 * E)
    x = torch.randn(tokens, K, device="cuda", generator=g).to(dt)
    w = (torch.randn(E, N, K, device="cuda", generator=g) * K ** -0.5).to(dt)
    rows = x[p.row.long()].contiguous()
    out = torch.empty(tokens * top, N, device="cuda", dtype=dt)
    for _ in range(2):
        X.product(rows, w, p, out, act)
    ids = X.route(logits, top)[0].reshape(-1)
    expert = torch.empty_like(ids)
    expert[p.where.reshape(-1).long()] = ids
    want = (rows.double()[:, None] * w[expert.long()].double()).sum(-1)
    if act == "relu2":
        want = want.clamp(min=0).pow(2)
    elif act:
        want = getattr(torch.nn.functional, act)(want)
    scale = want.pow(2).mean().sqrt() + want.abs()
    assert bool(((out.double() - want).abs() <= (K * 2.0 ** -22 + STEP[dt]) * scale).all())


def test_rows_planned_before_a_capture(cuda):
    """A tile list of the stream form used under capture: no counters in the graph, and replays
    equal the eager result."""
    from cake_amd.ops import experts as X
    from cake_amd.ops import gemm as G
    E, N, K = 16, 200, 264
    logits = torch.randn(20, E, device="cuda")
    p = X.plan(*X.route(logits, 2), E, torch.bfloat16)
    assert p.cfg == G.ROWS
    x = torch.randn(40, K, device="cuda").to(torch.bfloat16)
    w = (torch.randn(E, N, K, device="cuda") * K ** -0.5).to(torch.bfloat16)
    want = X.product(x, w, p, torch.empty(40, N, device="cuda", dtype=torch.bfloat16)).float()
    out = torch.empty(40, N, device="cuda", dtype=torch.bfloat16)
    before, graph = set(G._ticks), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        X.product(x, w, p, out)
    assert set(G._ticks) == before
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        torch.testing.assert_close(out.float(), want, rtol=2.0 ** -7, atol=2.0 ** -7)
        X.product(x, w, p, torch.empty_like(out))
