"""One token's mixer with the feed-forward's up rows beside it, against the two as launches of their own."""
import pytest
import torch

from cake_amd.ops import mixers as M

pytestmark = pytest.mark.gpu
HALF = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _up(g, dt, K, N, ln, kind):
    """Rows, and their result in 64 bits with the bound of a 16-bit one: the norm and K sums are f32."""
    width = K - 3 if K % 64 else K
    x, nw = torch.zeros(K), torch.zeros(K)
    x[:width], nw[:width] = torch.randn(width, generator=g) + 0.3, torch.randn(width, generator=g) * 0.1
    w = torch.randn(N, K, generator=g).mul(K ** -0.5).to(dt)
    act = torch.full((N + 8,), 7.0, device="cuda", dtype=dt)
    up = M.UpRows(x.cuda(), nw.to(dt).cuda(), 1e-5, 1.0, ln, width, w.cuda(), act[:N], kind)
    h = x.double()[:width]
    h = h - h.mean() if ln else h
    h = h * torch.rsqrt(h.pow(2).mean() + 1e-5) * (1 + nw.to(dt).double()[:width])
    y = w.double()[:, :width] @ h
    y = 0.5 * y * (1 + torch.erf(y / 2 ** 0.5)) if kind == "gelu" else y.clamp(min=0).pow(2)
    # of the sums (values of a few units, twice of it through the square), and a rounding to 16 bits
    return up, act, y, K * 2.0 ** -24 * 16 + 1.01 * HALF[dt] * y.abs()


def _check_up(up, act, y, tol):
    n = y.numel()
    assert ((up.act.cpu().double() - y).abs() <= tol).all()
    assert (act[n:] == 7).all()


# rows: fewer than a workgroup has waves, odd ones, several rounds of all waves; widths: both register forms,
# padded columns, a ragged end
@pytest.mark.parametrize("dt", list(HALF), ids=str)
@pytest.mark.parametrize("K,N,ln,kind", [(2048, 1, False, "gelu"), (2056, 11, True, "gelu"), (4096, 14001, False, "relu2"),
                                         (4104, 330, True, "relu2"), (8192, 515, False, "gelu")])
@pytest.mark.parametrize("H,G,dim,nsplit", [(16, 4, 128, 1), (18, 1, 64, 4), (32, 8, 120, 32)])
def test_attention(dt, K, N, ln, kind, H, G, dim, nsplit):
    g = torch.Generator().manual_seed(N + H)
    sh, S = M.AttnShape(H, G, dim, dim, 8), 1088
    assert M.takes_up_rows(sh, K)
    kc = torch.randn(2, G, S, sh.DP, generator=g).to(dt)
    vc = torch.randn(2, G, sh.DVP, S, generator=g).to(dt)
    kc[..., dim:], vc[:, :, dim:] = 0, 0
    proj = torch.randn(1, sh.qkv_cols + sh.out_cols, generator=g).cuda()
    cs = torch.randn(S, 16, generator=g).cuda()
    part = torch.zeros(sh.part_floats(1, nsplit), device="cuda")
    ticket = torch.zeros(sh.tiles, dtype=torch.int32, device="cuda")
    slot = torch.ones(1, dtype=torch.int32, device="cuda")
    for pos in (0, 33, 128, 255, 1087):
        p = torch.tensor([pos], dtype=torch.int32, device="cuda")
        got = []
        up, act, y, tol = _up(g, dt, K, N, ln, kind)
        for u in (None, up):
            k, v, out = kc.cuda(), vc.cuda(), torch.full((1, sh.out_cols + 8), 7.0, device="cuda", dtype=dt)
            M.attn_decode(sh, proj, p, slot, cs, True, True, True, 1e-5, 0.1, k, v, out, nsplit, part, ticket, u)
            got.append((out, k, v))
        _check_up(up, act, y, tol)
        (a, *ca), (b, *cb) = got
        assert all(torch.equal(s, t) for s, t in zip(ca, cb)) and int(ticket.abs().sum()) == 0
        # a split's keys lie in other waves: probabilities round elsewhere, half a unit each way, and the result
        d = (a.double() - b.double())[0, :sh.out_cols].norm() / a.double()[0, :sh.out_cols].norm()
        assert float(d) < 2 * HALF[dt], (pos, float(d))
        assert (b[0, sh.out_cols:] == 7).all()


@pytest.mark.parametrize("dt", list(HALF), ids=str)
@pytest.mark.parametrize("K,N,ln,kind", [(2048, 3, False, "gelu"), (4104, 11264, True, "relu2"), (8192, 700, False, "gelu")])
@pytest.mark.parametrize("H,G,dim,vdim,taps", [(16, 8, 128, 128, 4), (3, 1, 40, 70, 2), (64, 32, 64, 64, 5)])
def test_delta(dt, K, N, ln, kind, H, G, dim, vdim, taps):
    g = torch.Generator().manual_seed(N + H)
    sh = M.DeltaShape(H, G, dim, vdim, taps)
    assert M.takes_up_rows(sh, K)
    f = dict(generator=g)
    consts = dict(conv=torch.randn(taps, sh.channels, **f).cuda(), a_log=torch.randn(H, **f).cuda(),
                  dt_bias=torch.randn(H, **f).cuda(), norm_w=torch.randn(vdim, **f).cuda())
    state, ring = torch.randn(2, H, dim, sh.EP, **f), torch.randn(2, taps, sh.channels, **f)
    state[..., vdim:] = 0
    proj = torch.randn(1, sh.channels + sh.out_cols + 2 * H, **f).cuda()
    slot = torch.ones(1, dtype=torch.int32, device="cuda")
    for pos in (0, 1, 900):
        p = torch.tensor([pos], dtype=torch.int32, device="cuda")
        got = []
        up, act, y, tol = _up(g, dt, K, N, ln, kind)
        for u in (None, up):
            s, r, out = state.cuda(), ring.cuda(), torch.full((1, sh.out_cols + 8), 7.0, device="cuda", dtype=dt)
            M.delta_decode(sh, proj, proj[:, sh.channels + sh.out_cols:], p, slot, 1e-5, **consts, state=s, ring=r,
                           out=out, up=u)
            got.append((out, s, r))
        _check_up(up, act, y, tol)
        # the same body: fused multiply-adds may be chosen elsewhere, a few units of f32
        for a, b, t in zip(got[0], got[1], (HALF[dt], 1e-6, 0.0)):
            assert float((a.double() - b.double()).norm()) <= t * float(a.double().norm())


def test_what_stays_on_its_own():
    A, D = M.AttnShape, M.DeltaShape
    assert not M.takes_up_rows(A(16, 4, 128, 128), 1024) and not M.takes_up_rows(A(16, 4, 128, 128), 8200)
    assert not M.takes_up_rows(A(16, 4, 160, 160), 2048) and not M.takes_up_rows(A(16, 4, 128, 64), 2048)
    assert not M.takes_up_rows(D(4, 4, 256, 256, 4), 2048) and not M.takes_up_rows(D(257, 1, 64, 64, 4), 2048)
