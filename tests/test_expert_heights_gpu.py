"""Routed products whose tile height is chosen on the device (mixer_experts.hip, gemm_inst_grouped.hip): both k short, on the
four-wave tiles; long ones are in test_gemm_ws_gpu.py."""
import pytest
import torch

from cake_amd.ops import experts as X
from cake_amd.ops import gemm as G

pytestmark = pytest.mark.gpu


def _height(counts, F, W):
    """The rule in 64 bits: (cost, height) of every height."""
    ks, cols = (lambda k: -(-k // 64)), (lambda n: -(-n // 256))
    R, out = sum(counts), []
    mem = (len(counts) * F * W + R * (F + W)) * 2 / 8.2e6
    for bm, step, end in ((128, 1.106, 5.4), (160, 1.161, 7.76), (192, 1.38, 8.64), (256, 1.547, 11.64)):
        t = sum(-(-c // bm) for c in counts)
        out.append((max(-(-t * cols(F) // 256) * (step * ks(W) + end), mem)
                    + max(-(-t * cols(W) // 256) * (step * ks(F) + end), mem), bm))
    return out


# one group and many; even, skewed and empty ones, rows that end a tile of each height or pass it by one
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("counts,F,W", [([64], 72, 200), ([129, 128, 127, 1], 300, 136), ([160, 161, 0, 159, 97], 264, 520),
                                        ([192, 193, 191, 30], 1024, 256), ([256, 255, 257, 0, 512], 200, 72),
                                        ([100] * 60 + [150, 70, 0, 190], 1024, 512), ([190] * 64, 520, 1024)])
def test_height_of_the_groups(cuda, dt, counts, F, W):
    """The list holds the cheapest height (of two within 1e-4 either), and both products are one rounding
    (2^-8 or 2^-11) of f32 sums; nothing beside the rows is written."""
    E, R = len(counts), sum(counts)
    g = torch.Generator(device="cuda").manual_seed(R)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(R, generator=torch.Generator().manual_seed(1))]
    ids = ids.int().cuda().view(R, 1)
    p = X.plan(ids, torch.rand(R, 1, device="cuda", generator=g), E, dt, F * W, F)
    assert p.cfg == G.BY_LIST
    costs = _height(counts, F, W)
    bm = int(p.tiles[-1, 1])
    assert bm in [b for c, b in costs if c <= min(costs)[0] * (1 + 1e-4)]
    n = int(p.tiles[-1, 0])
    assert n == sum(-(-c // bm) for c in counts) and int(p.tiles[:n, 2].max()) <= bm
    x = torch.randn(R, W, device="cuda", generator=g).to(dt)
    up = (torch.randn(E, F, W, device="cuda", generator=g) * W ** -0.5).to(dt)
    out = torch.full((R, F + 8), 7.0, device="cuda", dtype=dt)
    X.product(x, up, p, out[:, :F], "relu2")
    r0, size = 0, 2.0 ** (-8 if dt == torch.bfloat16 else -11)
    for e, c in enumerate(counts):
        want = torch.relu(x[r0:r0 + c].float() @ up[e].float().t()).square()
        assert bool(((out[r0:r0 + c, :F].float() - want).abs() <= size * want + W * 2.0 ** -18 * (1 + want.sqrt())).all())
        r0 += c
    assert bool((out[:, F:] == 7.0).all())


def test_a_captured_plan_chooses_at_every_replay(cuda):
    """One graph, other groups at each replay: the height is the new ones'."""
    E, R, F, W = 8, 1600, 1024, 512
    ids = torch.zeros(R, 1, dtype=torch.int32, device="cuda")
    score = torch.ones(R, 1, device="cuda")
    x = torch.randn(R, W, device="cuda").bfloat16()
    up = (torch.randn(E, F, W, device="cuda") * W ** -0.5).bfloat16()
    out = torch.empty(R, F, device="cuda", dtype=torch.bfloat16)

    def step():
        p = X.plan(ids, score, E, torch.bfloat16, F * W, F)
        X.product(x, up, p, out, "relu2")
        return p.tiles
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        tiles = step()
    for counts in ([200] * 8, [1593] + [1] * 7, [130, 270] * 4, [256] * 6 + [64, 0]):
        ids.copy_(torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).int().view(R, 1))
        graph.replay()
        torch.cuda.synchronize()
        costs = _height(counts, F, W)
        assert int(tiles[-1, 1]) in [b for c, b in costs if c <= min(costs)[0] * (1 + 1e-4)]
        got = out.clone()
        step()
        assert torch.equal(got, out)
