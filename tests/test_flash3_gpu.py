"""Causal attention of 128-wide heads on the one-wave-per-SIMD core: row and key counts around its
tiles, cached prefixes, ragged batches, sink and gate, the latent form; against float64 and beside
the general kernel that takes what the core refuses."""
import pytest
import torch

from cake_amd.ops import hip as K
from cake_amd.ops import latent as L
from cake_amd.ops import mixers as M

pytestmark = pytest.mark.gpu

# the probabilities and the result are rounded once each, half a unit in the last place (the sums
# are float32)
TOL = {torch.bfloat16: 2 * 2 ** -8, torch.float16: 2 * 2 ** -11}
DTYPES = [torch.bfloat16, torch.float16]


def _want(q, k, v, pos0, scale, sink=False, gate=None):
    s = q.double() @ k.double().t().contiguous() * scale
    n, T = s.shape
    s.masked_fill_(torch.arange(T)[None] > torch.arange(n)[:, None] + pos0, float("-inf"))
    v = v.double()
    if sink:
        s = torch.cat([s, s.new_zeros(n, 1)], 1)
        v = torch.cat([v, v.new_zeros(1, v.shape[1])])
    o = s.softmax(1) @ v
    return o if gate is None else o * gate.double().sigmoid()


def _close(got, want, dt):
    assert bool(torch.isfinite(got).all())
    assert float((got.double() - want).norm() / want.norm()) < TOL[dt]


@pytest.mark.parametrize("dt", DTYPES, ids=str)
@pytest.mark.parametrize("H,Hkv,N,pos0", [
    (4, 2, 1, 0), (4, 1, 31, 33), (2, 2, 33, 0), (4, 2, 64, 64), (8, 8, 65, 3), (2, 1, 127, 1),
    (2, 1, 129, 191), (3, 1, 256, 0), (2, 2, 641, 0), (192, 8, 257, 0), (192, 64, 300, 21)])
def test_prefill(dt, H, Hkv, N, pos0):
    """The last two have the workgroups for 64 rows a wave; keys past the live ones are NaN."""
    g = torch.Generator().manual_seed(N)
    S, Tk = pos0 + N + 37, pos0 + N
    qkv = torch.randn(N, (H + 3) * 128, generator=g).to(dt)       # q is a column block of it
    kc, vc = (torch.randn(Hkv, S, 128, generator=g).to(dt) for _ in range(2))
    kc[:, Tk:], vc[:, Tk:] = float("nan"), float("nan")
    qd, kd, vd = qkv.cuda(), kc.cuda(), vc.cuda()
    out = torch.full((N + 1, H * 128), 7.0, device="cuda", dtype=dt)
    K.flash_attn(qd[:, :H * 128].view(1, N, H, 128).transpose(1, 2), kd[None, :, :Tk],
                 vd[None, :, :Tk], out[:N].view(1, N, H, 128).transpose(1, 2), 0.1, causal=True,
                 pos0=pos0)
    assert bool((out[N:] == 7.0).all())
    for h in sorted({0, H // 2, H - 1}):
        hk = h // (H // Hkv)
        _close(out[:N, h * 128:h * 128 + 128].cpu(),
               _want(qkv[:, h * 128:h * 128 + 128], kc[hk, :Tk], vc[hk, :Tk], pos0, 0.1), dt)


@pytest.mark.parametrize("dt", DTYPES, ids=str)
def test_prefill_batch_and_standing_out_key(dt):
    """Batched views; and a key far above the many others, whose share is of tiny probabilities."""
    q, k, v = (torch.randn(3, n, 70, 128).to(dt) for n in (4, 2, 2))
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    out = torch.empty_like(qd)
    K.flash_attn(qd, kd, vd, out, 0.2, causal=True)
    for b in range(3):
        _close(out[b, 3].cpu(), _want(q[b, 3], k[b, 1], v[b, 1], 0, 0.2), dt)
    n, d = 3000, 9.0
    q, k, v = torch.zeros(n, 128), torch.zeros(n, 128), torch.ones(n, 128)
    q[:, 0], k[n // 2, 0], v[n // 2] = 1, d, 0
    out = torch.empty(1, 1, n, 128, device="cuda", dtype=dt)
    K.flash_attn(q.to(dt).cuda()[None, None], k.to(dt).cuda()[None, None],
                 v.to(dt).cuda()[None, None], out, 1.0, causal=True)
    _close(out[0, 0].cpu(), _want(q, k, v, 0, 1.0), dt)


@pytest.mark.parametrize("dt", DTYPES, ids=str)
@pytest.mark.parametrize("sink,gated", [(True, True), (False, False)])
@pytest.mark.parametrize("H,G,seqs", [
    (8, 2, [(1, 0, 5), (0, 70, 300), (3, 0, 129)]), (4, 4, [(0, 0, 128), (2, 63, 1)]),
    (2, 1, [(0, 1, 641)])])
def test_ragged(dt, H, G, seqs, sink, gated):
    sh, S = M.AttnShape(H, G, 128, 128), 704
    rows = M.Rows.pack([(s, p, [0] * n) for s, p, n in seqs], "cuda")
    g = torch.Generator().manual_seed(H)
    kc, vc = (torch.randn(4, G, *d, generator=g).to(dt) for d in ((S, 128), (128, S)))
    qn = torch.randn(rows.N, H, 128, generator=g).to(dt)
    gate = torch.randn(rows.N, H * 128 + 8, generator=g).to(dt) if gated else None
    dev = [None if t is None else t.cuda() for t in (qn, kc, vc, gate)]
    outs = []
    for ld in (H * 128 + 4, H * 128 + 1):    # the core; rows off 8 bytes: the general kernel
        out = torch.full((rows.N, ld), 7.0, device="cuda", dtype=dt)
        M.attn_prompt(sh, dev[0], dev[1], dev[2], rows, dev[3][:, :H * 128] if gated else None,
                      out[:, :H * 128], 0.1, sink)
        assert bool((out[:, H * 128:] == 7.0).all())
        outs.append(out[:, :H * 128].cpu())
    for r0, n, p0, s in rows.host:
        for h in (0, H - 1):
            c, hk = slice(h * 128, h * 128 + 128), h // (H // G)
            w = _want(qn[r0:r0 + n, h], kc[s, hk, :p0 + n], vc[s, hk, :, :p0 + n].t(), p0, 0.1,
                      sink, gate[r0:r0 + n, c] if gated else None)
            for out in outs:
                _close(out[r0:r0 + n, c], w, dt)


@pytest.mark.parametrize("dt", DTYPES, ids=str)
@pytest.mark.parametrize("H,seqs", [(4, [(1, 0, 5), (0, 70, 300), (2, 0, 129)]), (2, [(0, 1, 513)])])
def test_latent(dt, H, seqs):
    S = 576
    sh = L.LatentShape(H, 128, 64, 128, 96, 64, 30)
    rows = M.Rows.pack([(s, p, [0] * n) for s, p, n in seqs], "cuda")
    g = torch.Generator().manual_seed(H)
    cache = torch.randn(3, S, sh.LD, generator=g).to(dt)
    k = torch.randn(rows.n_keys, H * 128, generator=g).to(dt)
    vt = torch.randn(H * 128, rows.n_keys, generator=g).to(dt)
    q = torch.randn(rows.N, H * 192, generator=g).to(dt)
    ang = torch.rand(S, 30, generator=g) * 6
    cs = torch.stack([ang.cos(), ang.sin()], 2).reshape(S, 60).contiguous()
    qd, kd, vd, cd, sd = (t.cuda() for t in (q, k, vt, cache, cs))
    outs = []
    for ld in (H * 128, H * 128 + 1):
        out = torch.full((rows.N, ld), 7.0, device="cuda", dtype=dt)
        L.prompt(sh, qd, kd, vd, rows, sd, cd, out[:, :H * 128], 0.08)
        outs.append(out[:, :H * 128].cpu())
    for i, (r0, n, p0, s) in enumerate(rows.host):
        k0 = int(rows.key0[i])
        for h in (0, H - 1):
            qq = q[r0:r0 + n, h * 192:h * 192 + 192].float()
            c, sn = ang[p0:p0 + n].cos(), ang[p0:p0 + n].sin()
            x, y = qq[:, 128:188:2].clone(), qq[:, 129:188:2].clone()
            qq[:, 128:188:2], qq[:, 129:188:2] = x * c - y * sn, y * c + x * sn
            kk = torch.cat([k[k0:k0 + p0 + n, h * 128:h * 128 + 128],
                            cache[s, :p0 + n, sh.RP:sh.RP + 64]], 1)
            w = _want(qq.to(dt), kk, vt[h * 128:h * 128 + 128, k0:k0 + p0 + n].t(), p0, 0.08)
            for out in outs:
                _close(out[r0:r0 + n, h * 128:h * 128 + 128], w, dt)


@pytest.mark.parametrize("dt", DTYPES, ids=str)
@pytest.mark.parametrize("n", [1, 12, 13, 32, 33])
def test_many_short_sequences(dt, n):
    """Either side of the lines between the core and the general kernel, in both forms."""
    H, B, S = 16, 17, 64
    rows = M.Rows.pack([(i, 0, [0] * (n - i % 2 * (n > 1))) for i in range(B)], "cuda")
    lat = L.LatentShape(H, 128, 64, 128, 96, 64, 30)
    g = torch.Generator().manual_seed(n)

    def rnd(*s):
        return torch.randn(*s, generator=g).to(dt)
    qn, kc, vc = rnd(rows.N, H, 128), rnd(B, 4, S, 128), rnd(B, 4, 128, S)
    lq, lk, vt, cache = rnd(rows.N, H * 192), rnd(rows.n_keys, H * 128), rnd(H * 128, rows.n_keys), rnd(B, S, lat.LD)
    cs = torch.tensor([1.0, 0.0], device="cuda").repeat(S, 30)   # no rotation
    out = torch.empty(2, rows.N, H * 128, device="cuda", dtype=dt)
    M.attn_prompt(M.AttnShape(H, 4, 128, 128), qn.cuda(), kc.cuda(), vc.cuda(), rows, None, out[0], 0.1, True)
    L.prompt(lat, lq.cuda(), lk.cuda(), vt.cuda(), rows, cs, cache.cuda(), out[1], 0.08)
    got = out.cpu()
    for i in (0, 9, B - 1):
        r0, m, _, s = rows.host[i]
        k0 = int(rows.key0[i])
        for h in (0, H - 1):
            c = slice(h * 128, h * 128 + 128)
            _close(got[0, r0:r0 + m, c],
                   _want(qn[r0:r0 + m, h], kc[s, h // 4, :m], vc[s, h // 4, :, :m].t(), 0, 0.1, True), dt)
            kk = torch.cat([lk[k0:k0 + m, c], cache[s, :m, lat.RP:lat.RP + 64]], 1)
            _close(got[1, r0:r0 + m, c],
                   _want(lq[r0:r0 + m, h * 192:h * 192 + 192], kk, vt[c, k0:k0 + m].t(), 0, 0.08), dt)


def _first_touched(n, p0, p, rows):
    """First of n rows at positions p0.. that a value of probability 0 at key p may reach: of the
    first wave (`rows` rows) that takes the key's run of `rows` keys."""
    return next(r for r in range(0, n, rows) if p // rows * rows <= p0 + r + rows - 1)


@pytest.mark.parametrize("dt", DTYPES, ids=str)
@pytest.mark.parametrize("H,Hkv,N,pos0,p,rows", [
    (2, 1, 300, 0, 96, 32), (2, 1, 300, 0, 127, 32), (2, 2, 300, 13, 201, 32), (2, 1, 129, 0, 128, 32),
    (192, 8, 300, 0, 192, 64), (192, 8, 300, 64, 290, 64)])
def test_non_finite_values_stay_behind_prefill(dt, H, Hkv, N, pos0, p, rows):
    """A row before an infinite or NaN value does not see it, save in the wave that takes its keys."""
    g = torch.Generator().manual_seed(p)
    q, k, v = (torch.randn(1, h, n, 128, generator=g).to(dt).cuda()
               for h, n in ((H, N), (Hkv, pos0 + N), (Hkv, pos0 + N)))
    clean, got = torch.empty_like(q), torch.empty_like(q)
    K.flash_attn(q, k, v, clean, 0.1, causal=True, pos0=pos0)
    for bad in (float("inf"), float("nan")):
        v[:, :, p] = bad
        K.flash_attn(q, k, v, got, 0.1, causal=True, pos0=pos0)
        first = _first_touched(N, pos0, p, rows)
        assert 0 < first < N
        assert torch.equal(got[:, :, :first], clean[:, :, :first])
        assert not bool(torch.isfinite(got[:, :, p - pos0:]).any())   # those that do see it


@pytest.mark.parametrize("dt", DTYPES, ids=str)
@pytest.mark.parametrize("p0,n,p", [(0, 300, 96), (0, 300, 130), (45, 129, 150)])
def test_non_finite_values_stay_behind_hybrid(dt, p0, n, p):
    """The same of the hybrid designs' form and the latent one; and values past a sequence's last run
    of 32 keys (what an earlier sequence left in the slot) reach no row."""
    sh, S = M.AttnShape(2, 1, 128, 128), 448
    lat = L.LatentShape(2, 128, 64, 128, 96, 64, 30)
    rows = M.Rows.pack([(0, p0, [0] * n)], "cuda")
    g = torch.Generator().manual_seed(p)

    def rnd(*s):
        return torch.randn(*s, generator=g).to(dt).cuda()
    qn, kc, vc = rnd(n, 2, 128), rnd(1, 1, S, 128), rnd(1, 1, 128, S)
    cache, lk, vt = rnd(1, S, lat.LD), rnd(rows.n_keys, 256), rnd(256, rows.n_keys)
    lq, cs = rnd(n, 2 * 192), torch.rand(S, 60, generator=g).cuda()

    def both():
        a = torch.empty(n, 256, device="cuda", dtype=dt)
        b = torch.empty_like(a)
        M.attn_prompt(sh, qn, kc, vc, rows, None, a, 0.1, True)
        L.prompt(lat, lq, lk, vt, rows, cs, cache, b, 0.08)
        return torch.stack([a, b])
    end = -(-(p0 + n) // 32) * 32
    vc[..., end:], vt[:, end:] = float("nan"), float("nan")
    clean = both()
    assert bool(torch.isfinite(clean).all())
    vc[..., p], vt[:, p] = float("inf"), float("nan")
    got, first = both(), _first_touched(n, p0, p, 32)
    assert first > 0 and torch.equal(got[:, :first], clean[:, :first])
    assert not bool(torch.isfinite(got[:, p - p0:]).any())


@pytest.mark.parametrize("sn", [64, 1 << 22])
def test_prefill_rows_outside_the_cores_offsets(sn):
    """Key and value rows that overlap, or lie 2 GB apart in all: the general kernel, as ever."""
    n, dt = 300, torch.bfloat16
    buf = torch.zeros((n - 1) * sn + 512, device="cuda", dtype=dt)
    rows = buf.as_strided((n, 512), (sn, 1))
    g = torch.Generator(device="cuda").manual_seed(3)
    for r in range(n) if sn < 512 else [slice(None)]:
        rows[r] = torch.randn(rows[r].shape, device="cuda", generator=g).to(dt)
    k, v = (rows[:, c:c + 256].unflatten(1, (2, 128)).permute(1, 0, 2)[None] for c in (0, 256))
    q = torch.randn(1, 4, n, 128, device="cuda", generator=g).to(dt)
    out = torch.empty_like(q)
    K.flash_attn(q, k, v, out, 0.1, causal=True)
    for h in range(4):
        _close(out[0, h].cpu(), _want(q[0, h].cpu(), k[0, h // 2].cpu(), v[0, h // 2].cpu(), 0, 0.1), dt)


def test_ragged_caches_outside_the_cores_offsets():
    """A sequence's keys or values of 2 GB, in the hybrid designs' form and the latent one."""
    n, dt, S = 200, torch.bfloat16, 1 << 23
    rows = M.Rows.pack([(0, 0, [0] * n)], "cuda")
    g = torch.Generator(device="cuda").manual_seed(4)

    def rnd(*s):
        return torch.randn(*s, device="cuda", generator=g).to(dt)
    kc, vc = (torch.zeros(1, 1, *d, device="cuda", dtype=dt) for d in ((S, 128), (128, S)))
    kc[0, 0, :n], vc[0, 0, :, :n], qn = rnd(n, 128), rnd(128, n), rnd(n, 1, 128)
    out = torch.empty(n, 128, device="cuda", dtype=dt)
    M.attn_prompt(M.AttnShape(1, 1, 128, 128), qn, kc, vc, rows, None, out, 0.1, True)
    _close(out.cpu(), _want(qn[:, 0].cpu(), kc[0, 0, :n].cpu(), vc[0, 0, :, :n].t().cpu(), 0, 0.1, True),
           dt)
    del kc, vc
    lat = L.LatentShape(1, 128, 64, 128, 96, 64, 30)
    cs = torch.tensor([1.0, 0.0], device="cuda").repeat(256, 30)   # no rotation
    vt = torch.zeros(128, (1 << 23) + 69632, device="cuda", dtype=dt)
    vt[:, :n], lk, q, cache = rnd(128, n), rnd(rows.n_keys, 128), rnd(n, 192), rnd(1, 256, lat.LD)
    L.prompt(lat, q, lk, vt, rows, cs, cache, out, 0.08)
    kk = torch.cat([lk[:n], cache[0, :n, lat.RP:lat.RP + 64]], 1).cpu()
    _close(out.cpu(), _want(q.cpu(), kk, vt[:, :n].t().cpu(), 0, 0.08), dt)
