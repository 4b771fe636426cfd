"""The sum over a token's experts and the norm behind it in one launch, against the two."""
import pytest
import torch

from cake_amd.ops import experts as X
from cake_amd.ops import mixers as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("ln", [False, True])
@pytest.mark.parametrize("N,top,W", [(1, 1, 8), (13, 6, 2048), (5, 9, 1000), (3, 8, 4096), (2, 32, 4104), (40, 2, 8192)])
def test_sum_and_norm(dt, ln, N, top, W):
    g = torch.Generator("cuda").manual_seed(top + W)
    ids = torch.randint(0, 40, (N, top), device="cuda", generator=g, dtype=torch.int32)
    p = X.plan(ids, torch.rand(N, top, device="cuda", generator=g), 40, dt)
    y = torch.randn(N * top, W + 8, device="cuda", generator=g).to(dt)[:, :W]
    x = torch.randn(N, W, device="cuda", generator=g)
    w = torch.randn(W, device="cuda", generator=g)
    want, h, out = x.clone(), torch.empty(N, W, device="cuda", dtype=dt), torch.empty(N, W, device="cuda", dtype=dt)
    X.gather_sum(y, p, W, 0.37, want)
    M.norm(want, w, 1.0, 1e-5, W, h, ln=ln)
    X.gather_sum_norm(y, p, W, 0.37, x, w, 1.0, 1e-5, ln, out)
    assert torch.equal(x, want)   # one order of sums
    # f32 norms in two orders of sums: the last place of the 16-bit result where they round apart
    last = 2.0 ** (-7 if dt == torch.bfloat16 else -10)
    assert ((out.float() - h.float()).abs() <= last * h.float().abs() + 1e-6).all()
