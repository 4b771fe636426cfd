"""Products that leave their sums in slabs, and the norm and rotation that add them up."""
import ctypes as C

import pytest
import torch

from cake_amd.ops import gemm as G

pytestmark = pytest.mark.gpu
DTS = [torch.bfloat16, torch.float16]


def _slabs(x, w, kind, cfg, parts):
    M, K = x.shape
    N = w.shape[0]
    ws = torch.full((parts * M * N + 64,), float("nan"), device="cuda")   # the end stays untouched
    st = torch.cuda.current_stream().cuda_stream
    n = G._lib().cake_gemm_slabs(G._DT[x.dtype], kind, cfg, parts, x.data_ptr(), K, w.data_ptr(), K,
                                 ws.data_ptr(), G._zeros16(x.device).data_ptr(), M, N, K, st)
    assert 1 <= n <= parts, n
    assert torch.isnan(ws[n * M * N:]).all()
    return ws, n


# k of whole steps and not, columns of whole strips and not, parts that do not divide the steps
@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("M,N,K,kind,cfg,parts", [
    (1, 64, 512, 2, 0, 1), (2, 132, 1032, 2, 0, 2), (5, 2048, 2048, 2, 0, 4), (16, 100, 1928, 2, 0, 3),
    (17, 256, 1096, 2, 0, 2), (24, 388, 3584, 2, 0, 5), (45, 1024, 4096, 2, 0, 8), (64, 132, 2056, 2, 0, 3),
    (33, 36 * 128, 512, 2, 0, 1), (7, 300, 776, 1, 0, 1), (32, 4100, 520, 1, 0, 1),
    (45, 260, 1024, 0, 13, 4), (70, 192, 1032, 0, 12, 2), (130, 128, 2048, 0, 7, 8)])
def test_slabs_sum_to_the_product(dt, M, N, K, kind, cfg, parts):
    g = torch.Generator("cuda").manual_seed(M + N)
    x = torch.randn(M, K, device="cuda", generator=g).to(dt)
    w = torch.randn(N, K, device="cuda", generator=g).to(dt)
    ws, n = _slabs(x, w, kind, cfg, parts)
    got = ws[:n * M * N].view(n, M, N).double().sum(0)
    ref = x.double() @ w.double().t()
    # exact products, K of them added in f32: at most K 2^-24 of the sum of magnitudes, far less in the mean
    assert (got - ref).norm() <= 4e-6 * ref.norm()


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("M,N,n", [(1, 64, 1), (3, 2048, 2), (24, 2052, 3), (45, 4096, 8), (2, 4100, 5),
                                   (5, 8192, 16), (300, 512, 4), (4, 512, 0)])
@pytest.mark.parametrize("ln,w32,biased,normed", [(0, 0, False, True), (0, 1, False, True), (1, 1, True, True),
                                                  (0, 0, True, False)])
def test_slab_norm(dt, M, N, n, ln, w32, biased, normed):
    g = torch.Generator("cuda").manual_seed(N + n)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    slabs, ldx = rnd(n, M, N), N + 8
    x, w, bias = rnd(M, ldx), rnd(N) + 1, rnd(N).to(dt)
    w = w if w32 else w.to(dt)
    out = torch.empty(M, N, device="cuda", dtype=dt)
    off, alpha, eps = 0.5, 0.75, 1e-5
    want = x.double()
    if n:
        want[:, :N] += alpha * (slabs.double().sum(0) + (bias.double() if biased else 0))
    got = x.clone()
    rc = G._lib().cake_slab_norm(G._DT[dt], slabs.data_ptr() if n else None, n, got.data_ptr(), ldx,
                                 bias.data_ptr() if biased else None, alpha, w.data_ptr() if normed else None,
                                 w32, off, eps, ln, M, N, out.data_ptr(), N,
                                 torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert torch.equal(got[:, N:], x[:, N:])
    # n + 2 additions in f32 of values of a few units
    assert (got.double() - want).abs().max() <= (n + 2) * 2.0 ** -20
    if normed:
        v = want[:, :N] - (want[:, :N].mean(-1, keepdim=True) if ln else 0)
        ref = v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + eps) * (off + w.double())
        half = 2.0 ** (-8 if dt == torch.bfloat16 else -11)   # of a last place, at most; the rest is f32
        assert ((out.double() - ref).abs() <= 1.01 * half * ref.abs() + 1e-5).all()


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("T,nh,nkv,hd,pos0,n", [(1, 1, 1, 8, 0, 1), (5, 16, 4, 128, 0, 2), (45, 32, 8, 128, 7, 8),
                                                (3, 4, 2, 64, 1000, 3), (2, 3, 1, 256, 0, 5), (9, 5, 1, 24, 3, 4)])
def test_slab_rope(dt, T, nh, nkv, hd, pos0, n):
    g = torch.Generator("cuda").manual_seed(hd + n)
    cols, S = (nh + 2 * nkv) * hd, pos0 + T + 2
    slabs = torch.randn(n, T, cols, device="cuda", generator=g)
    inv = 1.0 / 10000.0 ** (torch.arange(0, hd, 2, device="cuda") / hd)
    q = torch.zeros(T, cols, device="cuda", dtype=dt)
    kc, vc = (torch.zeros(nkv, S, hd, device="cuda", dtype=dt) for _ in range(2))
    rc = G._lib().cake_slab_rope(G._DT[dt], slabs.data_ptr(), n, q.data_ptr(), cols, T, nh, nkv, hd, inv.data_ptr(),
                                 pos0, S, kc.data_ptr(), vc.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    y = slabs.double().sum(0).view(T, nh + 2 * nkv, hd)
    # the angle is an f32 product, as in the rotation of a step
    a = ((torch.arange(T, device="cuda") + pos0).float()[:, None] * inv).double()[:, None]
    u, v = y[..., :hd // 2], y[..., hd // 2:]
    r = torch.cat([u * a.cos() - v * a.sin(), u * a.sin() + v * a.cos()], -1)
    half = 2.0 ** (-8 if dt == torch.bfloat16 else -11)   # of a last place, at most

    def near(got, ref):
        assert ((got.double() - ref).abs() <= 1.01 * half * ref.abs() + 1e-5).all()
    near(q[:, :nh * hd].view(T, nh, hd), r[:, :nh])
    assert (q[:, nh * hd:] == 0).all()   # keys and values go to the cache alone
    near(kc[:, pos0:pos0 + T].transpose(0, 1), r[:, nh:nh + nkv])
    near(vc[:, pos0:pos0 + T].transpose(0, 1), y[:, nh + nkv:])
    for c in (kc, vc):
        assert (c[:, :pos0] == 0).all() and (c[:, pos0 + T:] == 0).all()


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("T", [1, 2, 15, 16, 17, 31, 32, 33, 45, 48, 49, 64])
@pytest.mark.parametrize("nh,nkv,hd,n", [(4, 2, 64, 1), (8, 1, 128, 3), (16, 16, 128, 8), (5, 5, 64, 2)])
def test_slab_attn(dt, T, nh, nkv, hd, n):
    g = torch.Generator("cuda").manual_seed(hd + n + T)
    cols, S = (nh + 2 * nkv) * hd, 70
    slabs = torch.randn(n, T, cols, device="cuda", generator=g) * n ** -0.5
    inv = 1.0 / 10000.0 ** (torch.arange(0, hd, 2, device="cuda") / hd)
    outs, caches = [], []
    for _ in range(2):
        out = torch.full((T, nh * hd + 8), 7.0, device="cuda", dtype=dt)
        kc, vc = (torch.full((nkv, S, hd), 5.0, device="cuda", dtype=dt) for _ in range(2))
        rc = G._lib().cake_slab_attn(G._DT[dt], slabs.data_ptr(), n, out.data_ptr(), nh * hd + 8, T, nh, nkv, hd,
                                     inv.data_ptr(), S, kc.data_ptr(), vc.data_ptr(), hd ** -0.5,
                                     torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        outs.append(out)
        caches.append((kc, vc))
    assert torch.equal(*outs) and (outs[0][:, nh * hd:] == 7).all()
    # the cache of the rotation of its own, row for row
    q = torch.zeros(T, cols, device="cuda", dtype=dt)
    k2, v2 = (torch.full((nkv, S, hd), 5.0, device="cuda", dtype=dt) for _ in range(2))
    assert G._lib().cake_slab_rope(G._DT[dt], slabs.data_ptr(), n, q.data_ptr(), cols, T, nh, nkv, hd,
                                   inv.data_ptr(), 0, S, k2.data_ptr(), v2.data_ptr(),
                                   torch.cuda.current_stream().cuda_stream) == 0
    half = 2.0 ** (-8 if dt == torch.bfloat16 else -11)
    for a, b in zip(caches[0], (k2, v2)):
        assert ((a.double() - b.double()).abs() <= 2 * half * b.double().abs() + 1e-6).all()
        assert (a[:, T:] == 5).all()
    # and its rows' attention in 64 bits: probabilities and results are rounded once each
    Q = q[:, :nh * hd].double().view(T, nh, hd)
    K, V = (c[:, :T].double().transpose(0, 1).repeat_interleave(nh // nkv, 1) for c in caches[0])
    s = torch.einsum("qhd,khd->hqk", Q, K) * hd ** -0.5
    p = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device="cuda").triu(1), -float("inf")).softmax(-1)
    want = torch.einsum("hqk,khd->qhd", p, V).reshape(T, -1)
    size = torch.einsum("hqk,khd->qhd", p, V.abs()).reshape(T, -1)
    assert ((outs[0][:, :nh * hd].double() - want).abs() <= 1.05 * half * (want.abs() + size) + 2 * half * size).all()


def test_refused():
    z, st = torch.zeros(4096, device="cuda"), torch.cuda.current_stream().cuda_stream
    p = z.data_ptr()
    L = G._lib()
    for kind, cfg, parts, M, N, K in ((2, 0, 1, 65, 64, 512), (1, 0, 1, 33, 64, 512), (1, 0, 2, 4, 64, 512),
                                      (0, 22, 2, 4, 64, 512), (0, 13, 1, 4, 64, 512), (3, 0, 1, 4, 64, 512),
                                      (2, 0, 1, 4, 64, 12)):
        assert L.cake_gemm_slabs(0, kind, cfg, parts, p, K, p, K, p, p, M, N, K, st) < 0
    assert L.cake_slab_norm(0, p, 1, p, 6, None, 1.0, None, 0, 0.0, 1e-5, 0, 1, 6, None, 0, st) != 0
    assert L.cake_slab_norm(0, p, 1, p, 8196, None, 1.0, None, 0, 0.0, 1e-5, 0, 1, 8196, None, 0, st) != 0
    assert L.cake_slab_rope(0, p, 1, p, 64, 1, 1, 1, 12, p, 0, 4, p, p, st) != 0
    for T, nh, nkv, hd, S in ((65, 1, 1, 64, 70), (2, 3, 2, 64, 4), (2, 1, 1, 96, 4), (5, 1, 1, 64, 4)):
        assert L.cake_slab_attn(0, p, 1, p, nh * hd, T, nh, nkv, hd, p, S, p, p, 1.0, st) != 0
