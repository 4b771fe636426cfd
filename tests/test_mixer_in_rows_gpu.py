"""Input products of one token: few rows (a pair a workgroup), and up to a workgroup a CU."""
import pytest
import torch

from cake_amd.ops import mixers as M

pytestmark = pytest.mark.gpu


# odd and even rows to either side of each rule's ends; columns of whole and ragged rounds
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("N", [1, 2, 65, 1024, 1025, 2048, 2049, 2560, 2561])
@pytest.mark.parametrize("K", [1016, 1024, 1032, 2048, 2056, 3000, 4088, 4096])
@pytest.mark.parametrize("ln", [False, True])
def test_rows(cuda, dt, N, K, ln):
    """f32 dot products of f32 normed rows in another order: K 2^-22 of the scale; the activated rows rounded once."""
    g = torch.Generator(device="cuda").manual_seed(N + K)
    x = 2 * torch.randn(K, device="cuda", generator=g) + 0.5
    nw = torch.rand(K, device="cuda", generator=g).to(dt)
    w = torch.empty(N, K, device="cuda", dtype=dt).normal_(0, K ** -0.5, generator=g)
    n_raw = (N + 1) // 2
    out = torch.full((n_raw + 4,), 5.0, device="cuda")
    act = torch.full((N - n_raw + 4,), 5.0, device="cuda", dtype=dt)
    M.layer_in(x, nw, 1e-5, 1.0, K, w, n_raw, out[:n_raw], act[:N - n_raw], ln=ln)
    h = x.double() - (x.double().mean() if ln else 0)
    h = h * torch.rsqrt(h.square().mean() + 1e-5) * (1 + nw.double())
    want = w.double() @ h
    tol = K * 2.0 ** -22 * (1 + want.abs())
    assert bool(((out[:n_raw].double() - want[:n_raw]).abs() <= tol[:n_raw]).all()) and bool((out[n_raw:] == 5.0).all())
    a = want[n_raw:]
    a = torch.nn.functional.gelu(a)
    size = 2.0 ** (-8 if dt == torch.bfloat16 else -11)
    assert bool(((act[:N - n_raw].double() - a).abs() <= 2 * tol[n_raw:] + size * a.abs()).all())
    assert bool((act[N - n_raw:] == 5.0).all())


# every number of rounds that a pair has, their ends met and not
@pytest.mark.parametrize("N", [1025, 2049, 2560])
@pytest.mark.parametrize("K", [1536, 1544, 2552, 2560, 3064, 3072, 3576, 3584, 3592])
def test_rounds_of_a_pair(cuda, N, K):
    test_rows(cuda, torch.bfloat16, N, K, False)


# whole rounds of 512 columns past the ones asked for ahead, one to three over, and pieces of a round
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("K", [2048, 2056, 2560, 3072, 3584, 4096, 4104, 6144, 11776, 29696, 30200])
def test_rounds_left_over(cuda, dt, K):
    """The output products of one token: 16-bit columns, f32 sums in another order (K 2^-22 of the scale)."""
    from cake_amd.ops import hip as K32
    N = 37
    g = torch.Generator(device="cuda").manual_seed(K)
    a = torch.randn(K, device="cuda", generator=g).to(dt)
    w = torch.empty(N, K, device="cuda", dtype=dt).normal_(0, K ** -0.5, generator=g)
    x = torch.randn(N, device="cuda", generator=g)
    y = torch.empty(N, device="cuda")
    want = w.double() @ a.double()
    M.layer_out(a, w, 0.5, x, y)
    assert bool(((y.double() - x.double() - 0.5 * want).abs() <= K * 2.0 ** -22 * (1 + want.abs())).all())
    r = x.clone()
    K32.gemv(a, w, r, accumulate=True)
    assert bool(((r.double() - x.double() - want).abs() <= K * 2.0 ** -22 * (1 + want.abs())).all())


# columns of one and of two rounds, which are not asked for as left over
@pytest.mark.parametrize("K", [8, 504, 512, 520, 1016, 1024, 1032])
def test_up_to_two_rounds(cuda, K):
    test_rounds_left_over(cuda, torch.bfloat16, K)
