"""Sums of a split product's slabs and the rotation of prompt rows: whole and ragged threads."""
import pytest
import torch

from cake_amd.ops import reference as R

pytestmark = pytest.mark.gpu


# four slabs at a time: fewer, as many, one more, a remainder; rows of one thread, of a thread's remainder
# (1003, 6), of a block and one thread (1028), gated halves; out columns of a wider, odd row
@pytest.mark.parametrize("M,N,K,splits", [(3, 1028, 1024, 3), (45, 1003, 512, 4), (130, 6, 640, 5),
                                          (70, 2048, 2048, 16), (1, 16, 128, 2)])
@pytest.mark.parametrize("epi", ["store", "resid32", "store32", "add16", "gelu", "swiglu"])
@pytest.mark.parametrize("apart", [0, 3])
def test_slabs_sum_to_the_product(cuda, M, N, K, splits, epi, apart):
    """f32 sums of 16-bit products in another order, and one rounding of a 16-bit result (2^-8)."""
    from cake_amd.ops import gemm as G
    if epi == "swiglu" and N % 16:
        N = 48
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn(2 * N if epi == "swiglu" else N, K, device="cuda", generator=g) * K ** -0.5).to(torch.bfloat16)
    dt = torch.float32 if epi in ("resid32", "store32") else torch.bfloat16
    rows = torch.full((M, N + apart), 7.0, device="cuda", dtype=dt)
    held = torch.randn(M, N, device="cuda", generator=g).to(dt)
    want = x.double() @ w.double().t()
    kw = {}
    if epi == "resid32":
        rows[:, :N] = held
        kw["resid"] = rows[:, :N]
        want = want + held.double()
    elif epi == "store32":
        kw["resid"] = rows[:, :N]
    else:
        kw["out"] = rows[:, :N]
        if epi == "add16":
            kw["resid"] = held
            want = want + held.double()
        elif epi == "gelu":
            want = torch.nn.functional.gelu(want)
        elif epi == "swiglu":
            want = torch.nn.functional.silu(want[:, :N]) * want[:, N:]
    G.linear(x, w, epi=epi, cfg=0, splits=splits, **kw)
    tol = K * 2.0 ** -22 + (2.0 ** -18 if dt == torch.float32 else 2.0 ** -8)
    scale = want.pow(2).mean().sqrt() + want.abs()
    assert bool(((rows[:, :N].double() - want).abs() <= tol * scale).all())
    assert bool((rows[:, N:] == 7.0).all())


# 16-byte pieces of a token: a thread's two and no more (512), one more (520), two rounds and some
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("nh,nkv,hd", [(40, 8, 128), (41, 8, 128), (64, 8, 128), (33, 16, 256), (3, 1, 16)])
def test_rotated_rows_of_many_pieces(cuda, dt, nh, nkv, hd):
    """The result is one rounding of an f32 sum of two products: 2^-8 (bf16) or 2^-11 of their size."""
    from cake_amd.ops import hip as K_
    g = torch.Generator(device="cuda").manual_seed(nh)
    T, pos0, S = 5, 70, 80
    qkv = torch.randn(T, (nh + 2 * nkv) * hd, device="cuda", generator=g).to(dt)
    was = qkv.clone()
    q, k, v = qkv.split([nh * hd, nkv * hd, nkv * hd], dim=1)
    kc = torch.zeros(nkv, S, hd, device="cuda", dtype=dt)
    vc = torch.zeros_like(kc)
    invf = R.inv_freq(hd, 500000.0).to(cuda)
    at = torch.arange(pos0, pos0 + T, device="cuda")
    K_.rope_kv(q, k, v, invf, pos0, kc, vc)
    old = [p.reshape(T, -1, hd) for p in was.split([nh * hd, nkv * hd, nkv * hd], dim=1)]
    size = 2.0 ** (-8 if dt == torch.bfloat16 else -11)
    for got, src in ((q.reshape(T, nh, hd), old[0]), (kc[:, pos0:pos0 + T].transpose(0, 1), old[1])):
        far = (got.float() - R.rope(src.float(), at, invf)).abs()
        pair = src.float().abs() + src.float().abs().roll(hd // 2, -1)
        assert bool((far <= size * pair + 1e-6).all())
    assert torch.equal(vc[:, pos0:pos0 + T].transpose(0, 1), old[2])
    assert torch.equal(qkv[:, nh * hd:], was[:, nh * hd:])
