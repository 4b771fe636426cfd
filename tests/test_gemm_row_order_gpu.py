"""Both orders of a tile's rows (by the weights' row stride) give one product."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# strides 4096 and 8192 with all of k or a part of it; 4160, 2048 and 12288 the other way
@pytest.mark.parametrize("K,stride", [(4096, 4096), (704, 4096), (1024, 8192), (4160, 4160), (2048, 2048), (512, 12288)])
@pytest.mark.parametrize("cfg,splits", [(22, 1), (22, 3), (23, 1), (24, 2), (25, 1)])
@pytest.mark.parametrize("epi", ["store", "swiglu"])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_row_orders(cuda, K, stride, cfg, splits, epi, dt):
    """f32 sums in another order, and one rounding of the result: 2^-8 (bf16) or 2^-11."""
    from cake_amd.ops import gemm as G
    g = torch.Generator(device="cuda").manual_seed(K)
    M, N = 333, 1504
    x = torch.randn(M, stride, device="cuda", generator=g).to(dt)[:, :K]
    w = (torch.randn(N, stride, device="cuda", generator=g) * K ** -0.5).to(dt)[:, :K]
    want = x.double() @ w.double().t()
    if epi == "swiglu":
        want = torch.nn.functional.silu(want[:, :N // 2]) * want[:, N // 2:]
    y = G.linear(x, w, epi=epi, cfg=cfg, splits=splits)
    tol = K * 2.0 ** -22 + 2.0 ** (-8 if dt == torch.bfloat16 else -11)
    assert bool(((y.double() - want).abs() <= tol * (want.pow(2).mean().sqrt() + want.abs())).all())
