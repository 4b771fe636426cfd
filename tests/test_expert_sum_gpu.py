"""The sum over a token's experts."""
import pytest
import torch

from cake_amd.ops import experts as X

pytestmark = pytest.mark.gpu


# eight rows at once: one, fewer, as many, a remainder; whole and ragged columns, odd rows of x
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("top", [1, 6, 8, 9, 32])
@pytest.mark.parametrize("W,apart,at", [(2048, 0, 0), (1026, 0, 0), (7, 1, 0), (1040, 4, 1), (3, 0, 0)])
def test_sum_over_a_tokens_experts(cuda, dt, top, W, apart, at):
    """f32 sums in the choices' order, one fused step onto x: within half a unit of the step's operands."""
    N, E = 5, 40
    g = torch.Generator(device="cuda").manual_seed(top + W)
    ids = torch.randint(0, E, (N, top), device="cuda", generator=g, dtype=torch.int32)
    p = X.plan(ids, torch.rand(N, top, device="cuda", generator=g), E, dt)
    pitch = (W + 3) // 4 * 4
    y = torch.randn(N * top, pitch, device="cuda", generator=g).to(dt)
    whole = torch.randn(N * (W + apart) + at, device="cuda", generator=g)
    was = whole.clone()
    x, old = (t[at:].view(N, W + apart)[:, :W] for t in (whole, was))
    X.gather_sum(y[:, :W], p, W, 0.37, x)
    s = torch.zeros(N, W, device="cuda")
    for k in range(top):
        s += y[p.where[:, k].long(), :W].float()
    alpha = torch.tensor(0.37).double().float().double()
    want = old.double() + alpha.item() * s.double()
    assert bool(((x.double() - want).abs() <= 2.0 ** -24 * (old.abs() + s.abs()).double()).all())
    rest = whole[at:].view(N, W + apart)[:, W:]
    assert torch.equal(rest, was[at:].view(N, W + apart)[:, W:]) and torch.equal(whole[:at], was[:at])
