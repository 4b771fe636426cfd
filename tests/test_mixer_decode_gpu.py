"""Decode attention of the hybrid designs: batches that get fewer key splits than asked for, live
lengths around a wave's and a workgroup's keys, against float64."""
import pytest
import torch

from cake_amd.ops import mixers as M

pytestmark = pytest.mark.gpu

# probabilities and result are rounded once each (half a unit in the last place), sums are float32
TOL = {torch.bfloat16: 2 * 2 ** -8, torch.float16: 2 * 2 ** -11, torch.float32: 1e-5}


@pytest.mark.parametrize("dt", list(TOL), ids=str)
@pytest.mark.parametrize("H,G,dim,B,nsplit", [
    (4, 2, 128, 1, 1), (4, 2, 128, 1, 4), (16, 4, 128, 70, 32), (2, 2, 64, 140, 8),
    (18, 1, 48, 9, 32), (4, 1, 160, 3, 1)])
def test_lengths(dt, H, G, dim, B, nsplit):
    sh, S = M.AttnShape(H, G, dim, dim), 576
    g = torch.Generator().manual_seed(B + nsplit)
    kc = torch.randn(B, G, S, sh.DP, generator=g).to(dt)
    vc = torch.randn(B, G, sh.DVP, S, generator=g).to(dt)
    kc[..., dim:], vc[:, :, dim:] = 0, 0
    proj = torch.randn(B, sh.qkv_cols + sh.out_cols, generator=g)
    lens = [1, 2, 31, 32, 33, 64, 65, 128, 129, 255, 256, 257, 288, 289, 512, 513, 576]
    part = torch.zeros(sh.part_floats(B, nsplit), device="cuda")
    ticket = torch.zeros(B * sh.tiles, dtype=torch.int32, device="cuda")
    pd, cs = proj.cuda(), torch.zeros(S, 0, device="cuda")
    for rep in range(3 if B < 4 else 1):
        tk = [lens[(i + 7 * rep) % len(lens)] for i in range(B)]
        pos = torch.tensor([t - 1 for t in tk], dtype=torch.int32, device="cuda")
        kd, vd = kc.cuda(), vc.cuda()
        out = torch.full((B, sh.out_cols), 7.0, device="cuda", dtype=dt)
        M.attn_decode(sh, pd, pos, torch.arange(B, dtype=torch.int32, device="cuda"), cs, False,
                      True, True, 1e-5, 0.1, kd, vd, out, nsplit, part, ticket)
        assert int(ticket.abs().sum()) == 0
        q, k, v, gate = proj.split([H * dim, G * dim, G * dim, H * dim], 1)
        q, k, v = (t.to(dt).double() for t in (q, k, v))
        for b in range(B):
            n = tk[b] - 1
            for h in (0, H - 1):
                hk, c = h // (H // G), slice(h * dim, h * dim + dim)
                kk = torch.cat([kc[b, hk, :n, :dim].double(), k[b:b + 1, hk * dim:hk * dim + dim]])
                vv = torch.cat([vc[b, hk, :dim, :n].t().double(), v[b:b + 1, hk * dim:hk * dim + dim]])
                s = torch.cat([kk @ q[b, c] * 0.1, torch.zeros(1, dtype=torch.double)])
                w = s.softmax(0)[:-1] @ vv * gate[b, c].double().sigmoid()
                assert float((out[b, c].cpu().double() - w).norm() / w.norm()) < TOL[dt], (b, h, n)
            assert torch.equal(kd[b, :, n, :dim].cpu().double().reshape(-1), k[b])
