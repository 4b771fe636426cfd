"""Output and gated products of up to eight narrow rows (gemm_few.hip)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
SIZE = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


# one row, a group of four and one more, all; k of a lane, amid a chunk of 128, of one round of eight chunks and past it, the
# most; one weight row, a group and one more, several groups a workgroup
@pytest.mark.parametrize("dt", list(SIZE), ids=str)
@pytest.mark.parametrize("M", [1, 4, 5, 8])
@pytest.mark.parametrize("N,K", [(1, 8), (5, 136), (4100, 1024), (2051, 1160), (520, 3072), (2048, 4096)])
def test_products(cuda, dt, M, N, K):
    """Against f32 sums in another order (K 2^-21 of the scale); the gated product's rows are normed in f32 and rounded
    once, its result too (a factor's error 2^-8 or 2^-11 on x shows as sqrt(K) of it in a sum: 8 for the tail).  Nothing
    beside the rows is written, and again gives the same bits."""
    from cake_amd.ops import gemm as G
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K + 8, device="cuda", generator=g).to(dt)[:, :K]
    w = torch.empty(N, K, device="cuda", dtype=dt).normal_(0, K ** -0.5, generator=g)
    outs = []
    for _ in range(2):
        r = torch.full((M, N + 4), 3.0, device="cuda")
        G.few_add(x, w, r[:, :N])
        assert bool((r[:, N:] == 3.0).all())
        outs.append(r)
    want = 3.0 + x.float() @ w.float().t()
    assert torch.equal(*outs) and bool(((outs[0][:, :N] - want).abs() <= K * 2.0 ** -20 + 2.0 ** -21 * want.abs()).all())
    if K > 3072:
        with pytest.raises(RuntimeError):
            G.few_gated(torch.zeros(M, K, device="cuda"), w[0].contiguous(), 1e-5, torch.zeros(2, K, device="cuda", dtype=dt),
                        torch.empty(M, 1, device="cuda", dtype=dt))
        return
    h = 3 * torch.randn(M, K + 4, device="cuda", generator=g)[:, :K]
    ln = torch.empty(K, device="cuda", dtype=dt).uniform_(0.5, 1.5, generator=g)
    w2 = torch.empty(2 * N, K, device="cuda", dtype=dt).normal_(0, K ** -0.5, generator=g)
    outs = []
    for _ in range(2):
        out = torch.full((M, N + 8), 7.0, device="cuda", dtype=dt)
        G.few_gated(h, ln, 1e-5, w2, out[:, :N])
        assert bool((out[:, N:] == 7.0).all())
        outs.append(out)
    n = (h * torch.rsqrt(h.square().mean(1, keepdim=True) + 1e-5) * ln.float()).to(dt).float()
    y = n @ w2.float().t()
    want = torch.nn.functional.silu(y[:, :N]) * y[:, N:]
    # a norm's last bit may fall the other way: one step of single elements of x, of weights around K^-1/2
    tol = SIZE[dt] * (want.abs() + 8 * K ** -0.5 * (1 + y[:, :N].abs() + y[:, N:].abs())) + K * 2.0 ** -20
    assert torch.equal(*outs) and bool(((outs[0][:, :N].float() - want).abs() <= tol).all())


@pytest.mark.parametrize("dt", list(SIZE), ids=str)
def test_not_a_number(cuda, dt):
    """A row of infinities and NaN leaves the others alone, as do weights past an odd k."""
    from cake_amd.ops import gemm as G
    x = torch.ones(3, 72, device="cuda", dtype=dt)
    x[1] = float("inf")
    x[1, 5] = float("nan")
    w = torch.ones(6, 80, device="cuda", dtype=dt)
    w[:, 72:] = float("nan")
    r = torch.zeros(3, 6, device="cuda")
    G.few_add(x, w[:, :72], r)
    assert bool((r[0] == 72).all()) and bool((r[2] == 72).all()) and bool(r[1].isnan().all())
    h = torch.ones(3, 72, device="cuda")
    h[1] = float("nan")
    out = G.few_gated(h, torch.ones(72, device="cuda", dtype=dt), 0.0, w[:, :72], torch.empty(3, 3, device="cuda", dtype=dt))
    want = (72 * torch.nn.functional.silu(torch.tensor(72.0))).to(dt).item()
    assert bool((out[0] == want).all()) and bool((out[2] == want).all()) and bool(out[1].isnan().all())
