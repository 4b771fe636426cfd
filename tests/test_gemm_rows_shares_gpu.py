"""Products of few rows in the stream form: every way its shares can fall on the strips."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# whole strips, several of them a workgroup, equal parts of one, ends anywhere; a last strip of one row
@pytest.mark.parametrize("M", [1, 16, 17, 45, 64])
@pytest.mark.parametrize("N,K", [(28672, 512), (32000, 1024), (1, 4096), (129, 8), (6144, 4096), (513, 2056),
                                 (2048, 8192), (4096, 3648), (70000, 192)])
@pytest.mark.parametrize("epi", ["store32", "swiglu"])
def test_shares(cuda, monkeypatch, M, N, K, epi):
    """f32 sums of 16-bit products in two orders (either within K 2^-22 of the sums' scale of the exact
    one: K 2^-21 apart), then 2^-16 for the f32 result (alpha and the oracle's own rounding) or one
    rounding to bf16, 2^-8; a second launch finds clean counters, the same bits."""
    from cake_amd.ops import gemm as G
    monkeypatch.setattr(G, "rows_kind", lambda *a: 2)
    if epi == "swiglu":
        N = max(32, N // 32 * 32)
    g = torch.Generator(device="cuda").manual_seed(N + M)
    x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).to(torch.bfloat16)
    y = x.float() @ w.float().t()
    if epi == "swiglu":
        y = torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:]
    outs = []
    for _ in range(2):
        kw = {"resid": torch.empty(M, N, device="cuda")} if epi == "store32" else {}
        outs.append(G.linear(x, w, epi=epi, **kw))
    assert torch.equal(outs[0], outs[1])
    tol = K * 2.0 ** -21 + (2.0 ** -16 if epi == "store32" else 2.0 ** -8)
    scale = y.pow(2).mean().sqrt() + y.abs()
    assert bool(((outs[0].float() - y).abs() <= tol * scale).all())
