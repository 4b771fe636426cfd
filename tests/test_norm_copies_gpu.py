"""Rows normed once and written to several places (mixer_rows.hip) against the gathered form."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32], ids=str)
@pytest.mark.parametrize("ln", [False, True])
@pytest.mark.parametrize("W,copies", [(8, 1), (1020, 3), (2048, 6), (2056, 2), (4096, 32), (8192, 4), (9000, 5)])
def test_copies_are_the_gathered_rows(cuda, dt, ln, W, copies):
    """Either side of every register width, one place and the most: the same sums, the same bits.
    Against 64 bits one rounding to the type, and of the difference from the mean half a unit of the
    largest |x| (16) and of the mean, over the deviation (3) times weight and scale (1.75): 2^-18."""
    from cake_amd.ops import mixers as M
    N, ld = 13, M.pad_to(W, 8)
    g = torch.Generator().manual_seed(W + copies)
    x = torch.zeros(N, ld)
    x[:, :W] = torch.randn(N, W, generator=g) * 3 + 1
    w = torch.zeros(ld)
    w[:W] = torch.rand(W, generator=g) + 0.5
    where = torch.randperm(N * copies, generator=g).view(N, copies).int()
    rows = torch.empty(N * copies, dtype=torch.int32)
    rows[where.flatten().long()] = torch.arange(N, dtype=torch.int32).repeat_interleave(copies)
    x, w, where, rows = (t.to(cuda) for t in (x, w, where, rows))
    scale = torch.rand(N * copies, generator=g).to(cuda)
    a, b = (torch.full((N * copies, ld), 7.0, dtype=dt, device=cuda) for _ in range(2))
    M.norm(x, w, 0.25, 1e-5, W, a, where=where, ln=ln, scale=scale)
    M.norm(x, w, 0.25, 1e-5, W, b, rows=rows, ln=ln, scale=scale)
    assert torch.equal(a, b)
    y = x[:, :W].double()
    y = y - y.mean(1, keepdim=True) if ln else y
    y = y * torch.rsqrt(y.pow(2).mean(1, keepdim=True) + 1e-5) * (0.25 + w[:W].double())
    want = y[rows.long()] * scale.double()[:, None]
    eps = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -20}[dt]
    assert bool(((a[:, :W].double() - want).abs() <= eps * want.abs() + 2.0 ** -18).all())
    assert not bool(a[:, W:].any())
