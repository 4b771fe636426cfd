"""The choice of few rows and their plan in one launch, against the two launches."""
import pytest
import torch

from cake_amd.ops import experts as X

pytestmark = pytest.mark.gpu


# a wave's row and two, the last of each; one block of logits, four, sixteen; plans by tiles, in the stream form
# and of 32 bits; strided logits
@pytest.mark.parametrize("N,E,top", [(1, 1, 1), (1, 64, 6), (13, 64, 6), (16, 1024, 32), (16, 65, 9), (17, 64, 6),
                                     (32, 64, 32), (32, 3, 2), (17, 65, 4), (33, 64, 6), (16, 256, 1), (2, 257, 32)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32], ids=str)
def test_one_launch_plans_as_two(cuda, monkeypatch, dt, N, E, top):
    g = torch.Generator(device="cuda").manual_seed(N + E)
    logits = torch.randn(N, E + 5, device="cuda", generator=g)[:, :E]
    logits[N // 2, :] = logits[N // 2, 0].clone()   # ties: the smaller index
    ids, score = X.route(logits, top)
    alone, calls = X.plan(ids, score, E, dt, 1 << 20, 1 << 10), []
    route = X.route
    monkeypatch.setattr(X, "route", lambda *a: calls.append(1) or route(*a))
    p = X.route_plan(logits, top, dt, 1 << 20, 1 << 10)
    assert bool(calls) == (N > (32 if E <= 64 else 16))
    assert p.cfg == alone.cfg and p.tiles.shape == alone.tiles.shape
    n = int(alone.tiles[-1, 0])
    assert torch.equal(p.tiles[:n], alone.tiles[:n]) and torch.equal(p.tiles[-1, :2], alone.tiles[-1, :2])
    # an expert's rows in any order, each with its entry's score, bit for bit
    assert torch.equal(p.scale[p.where.long()], score)
    assert torch.equal(p.where.flatten().sort().values, torch.arange(N * top, device="cuda", dtype=torch.int32))
    first = torch.bincount(ids.flatten().long(), minlength=E).cumsum(0)
    owner = torch.searchsorted(first, p.where.long().contiguous(), right=True)
    assert torch.equal(owner.int(), ids)
