"""The scan of the gated delta rule under load: more workgroups than the chip holds, sequences of every few chunks."""
import pytest
import torch

from cake_amd.ops import mixers as M

pytestmark = pytest.mark.gpu


# rows of one wave's share to the most, columns of whole blocks and not; one to five chunks, their ends met and not
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32], ids=str)
@pytest.mark.parametrize("H,G,dim,vdim", [(32, 16, 128, 128), (24, 8, 64, 72), (8, 8, 192, 100), (8, 4, 256, 256)])
def test_batch_is_its_sequences(cuda, dt, H, G, dim, vdim):
    """A sequence's read-outs and state are the same bits alone and among others, and again."""
    sh = M.DeltaShape(H, G, dim, vdim, 4)
    g = torch.Generator(device="cuda").manual_seed(dim)

    def rnd(*s, scale=1.0):
        return torch.randn(*s, device="cuda", generator=g) * scale
    const = [rnd(4, sh.channels, scale=0.5), torch.linspace(-4.0, 2.0, H, device="cuda"), rnd(H), 1 + rnd(vdim, scale=0.2)]
    lens = [1, 15, 16, 17, 31, 32, 33, 48, 49, 64, 65, 80] * 2
    data = [(rnd(n, sh.channels + sh.out_cols).to(dt), rnd(n, 2 * H)) for n in lens]

    def run(which):
        state = torch.full((len(lens), H, dim, sh.EP), 5.0, device="cuda")
        ring = torch.full((len(lens), 4, sh.channels), -3.0, device="cuda")
        rows = M.Rows.pack([(i, 0, [0] * lens[i]) for i in which], cuda)
        out = torch.empty(rows.N, sh.out_cols, device="cuda", dtype=dt)
        M.delta_prompt(sh, torch.cat([data[i][0] for i in which]), torch.cat([data[i][1] for i in which]), rows, 1e-5,
                       *const, state, ring, out)
        return out.split([lens[i] for i in which]), state, ring
    outs, state, ring = run(range(len(lens)))
    again = run(range(len(lens)))
    assert all(torch.equal(a, b) for a, b in zip(outs, again[0]))
    assert torch.equal(state, again[1]) and torch.equal(ring, again[2])
    for i in range(12):
        one, s, r = run([i])
        assert torch.equal(one[0], outs[i]) and torch.equal(s[i], state[i]) and torch.equal(r[i], ring[i]), lens[i]
        assert bool(torch.isfinite(one[0]).all())


# by the number of workgroups alone, of rows that fit more of them to a CU, of up to three chunks; of one chunk each
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32], ids=str)
@pytest.mark.parametrize("dim,vdim", [(64, 256), (128, 128), (192, 250), (256, 256)])
@pytest.mark.parametrize("longest", [16, 48])
def test_many_sequences_run_as_one(cuda, dt, dim, vdim, longest):
    """Both scans give the same bits: sequences among so many that the other kernel takes them, and alone."""
    H, G, B = 32, 16, 40
    sh = M.DeltaShape(H, G, dim, vdim, 4)
    g = torch.Generator(device="cuda").manual_seed(dim + longest)

    def rnd(*s, scale=1.0):
        return torch.randn(*s, device="cuda", generator=g) * scale
    const = [rnd(4, sh.channels, scale=0.5), torch.linspace(-4.0, 2.0, H, device="cuda"), rnd(H), 1 + rnd(vdim, scale=0.2)]
    lens = [1 + (7 * i + 15) % longest for i in range(B)]
    lens[3] = longest
    data = [(rnd(n, sh.channels + sh.out_cols).to(dt), rnd(n, 2 * H)) for n in lens]

    def run(which):
        state = torch.full((B, H, dim, sh.EP), 5.0, device="cuda")
        ring = torch.full((B, 4, sh.channels), -3.0, device="cuda")
        rows = M.Rows.pack([(i, 0, [0] * lens[i]) for i in which], cuda)
        out = torch.empty(rows.N, sh.out_cols, device="cuda", dtype=dt)
        M.delta_prompt(sh, torch.cat([data[i][0] for i in which]), torch.cat([data[i][1] for i in which]), rows, 1e-5,
                       *const, state, ring, out)
        return out.split([lens[i] for i in which]), state, ring
    outs, state, ring = run(range(B))
    for some in (range(2, 5), [17], [39]):
        one, s, r = run(some)
        for i, o in zip(some, one):
            assert torch.equal(o, outs[i]) and torch.equal(s[i], state[i]) and torch.equal(r[i], ring[i]), lens[i]
            assert bool(torch.isfinite(o).all())
