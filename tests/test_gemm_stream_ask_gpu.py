"""The stream form's asking waves (gemm_rows.h): strips' ends amid shares, cold weights, counters left clean."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# shares that end anywhere, in equal parts and in whole strips; one row of a tile and all four; ragged columns and k
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("M", [1, 16, 17, 48, 64])
@pytest.mark.parametrize("N,K", [(40, 6152), (1000, 8192), (9000, 4104), (4096, 14336), (33000, 1032)])
def test_stream_shares(cuda, dt, M, N, K):
    """f32 sums of 16-bit products in two orders (K 2^-21 of the scale) on a sum of its own; the same bits five
    times over weights that no cache holds, with other products between; every arrival counter is zero behind them."""
    from cake_amd.ops import _lib as L
    from cake_amd.ops import gemm as G
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(M + N)
    x = torch.randn(M, K, device=dev, generator=g).to(dt)
    w = torch.empty(N, K, device=dev, dtype=dt).normal_(0, K ** -0.5, generator=g)
    want = x.float() @ w.float().t() + 2.0
    flush = torch.empty(512 << 20, dtype=torch.uint8, device=dev)
    ws, tick = G._rows_state(dev, M, torch.cuda.current_stream().cuda_stream)
    first = None
    for _ in range(5):
        flush.add_(1)
        y = torch.full((M, N + 4), 2.0, device=dev)
        L.check(G._lib().cake_gemm_rows(0 if dt == torch.bfloat16 else 1, G.EPI["resid32"], 2, x.data_ptr(), K,
                                        w.data_ptr(), K, None, 0, None, y.data_ptr(), N + 4, ws.data_ptr(),
                                        tick.data_ptr(), G._zeros16(x.device).data_ptr(), M, N, K, 1.0,
                                        torch.cuda.current_stream().cuda_stream), "rows")
        assert not bool(tick.any()) and bool((y[:, N:] == 2.0).all())
        first = y if first is None else first
        assert torch.equal(y, first)
    assert bool(((first[:, :N] - want).abs() <= K * 2.0 ** -20 + 2.0 ** -21 * want.abs()).all())
