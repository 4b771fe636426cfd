"""A layer's projections as one product by sections of columns, against the plain product."""
import pytest
import torch

from cake_amd.ops import gemm as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 2, 16, 17, 45, 64])
# sections that end amid a strip, amid a 16-row fragment, empty ones; strips in parts and whole
@pytest.mark.parametrize("n1,n2,N,K", [(0, 640, 1664, 1024), (384, 452, 1200, 520), (260, 260, 4104, 2048),
                                       (0, 0, 128, 512), (132, 388, 388, 1032), (10240, 10304, 29760, 512)])
def test_sections(monkeypatch, dt, M, n1, n2, N, K):
    monkeypatch.setattr(G, "rows_kind", lambda *a: 2)
    g = torch.Generator("cuda").manual_seed(N + M)
    x = torch.randn(M, K, device="cuda", generator=g).to(dt)
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).to(dt)

    def room(n, t, ld):   # rows further apart than their columns, the room between them untouched
        full = torch.full((M, n + ld), 7.0, device="cuda", dtype=t)
        return full, full[:, :n]
    (f16, o16), (f32, o32), (fa, act) = room(n1, dt, 8), room(n2 - n1, torch.float32, 4), room(N - n2, dt, 16)
    for _ in range(2):   # the second launch finds clean counters
        assert G.sections(x, w, n1, n2, o16, o32, act)
    y = x.double() @ w.double().t()
    half = 2.0 ** (-8 if dt == torch.bfloat16 else -11)
    gelu = 0.5 * y * (1 + torch.erf(y / 2 ** 0.5))
    sums = K * 2.0 ** -24 * 4   # K f32 sums of values of a few units
    for got, ref, tol in ((o16, y[:, :n1], half), (o32, y[:, n1:n2], 0.0), (act, gelu[:, n2:], half)):
        if ref.numel():
            assert ((got.double() - ref).abs() <= 1.01 * tol * ref.abs() + sums + 4e-7).all()
    for full, n in ((f16, n1), (f32, n2 - n1), (fa, N - n2)):
        assert (full[:, n:] == 7).all()


def test_left_to_the_separate_products():
    x, w = torch.zeros(4, 64, device="cuda").half(), torch.zeros(30, 64, device="cuda").half()
    out = torch.zeros(4, 30, device="cuda").half()
    assert not G.sections(x, w, 30, 30, out, None, None)          # a section amid a group of four
    assert not G.sections(torch.zeros(65, 64, device="cuda").half(), w[:28], 0, 0, None, None, out)
