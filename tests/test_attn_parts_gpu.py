"""Decode attention with a kv head's group in parts (attention.hip attn2_parts_kernel)."""
import math

import pytest
import torch

from cake_amd.ops import hip as K
from cake_amd.ops import reference as R

pytestmark = pytest.mark.gpu


# two parts of two, halves and quarters of eight; launches for short and long contexts, in turns over one workspace
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("nh,nkv,hd", [(32, 8, 128), (64, 8, 128), (8, 1, 64), (4, 1, 128)])
def test_launches_in_turns(cuda, dt, nh, nkv, hd):
    """Merged splits are this launch's own, whichever launch wrote the workspace before; a keys' block's ends; f32 attention
    within a rounding of 16-bit queries and result."""
    g = torch.Generator(device="cuda").manual_seed(nh)
    S = 2048
    kc = torch.randn(nkv, S, hd, device="cuda", generator=g).to(dt)
    vc = torch.randn(nkv, S, hd, device="cuda", generator=g).to(dt)
    part = torch.zeros(K.attn_workspace_numel(nh, hd, S), device="cuda")
    tickets = torch.zeros(2 * nkv + 2, dtype=torch.int32, device="cuda")
    out = torch.empty(nh * hd, device="cuda", dtype=dt)
    size = 2.0 ** (-7 if dt == torch.bfloat16 else -10)
    prev = K._ATTN_SINGLE[0]
    K.attn_set_single_max(0)   # short contexts take the split and merge path too
    try:
        for turn, (cap, pos) in enumerate([(8, 100), (8, 101), (8, 300), (0, 300), (0, 1500), (8, 102), (0, 65), (8, 300),
                                           (8, 15), (8, 16), (0, 2047), (0, 0), (8, 500), (8, 300), (0, 300), (8, 300)]):
            K.check(K.kernels().cake_attn_set_split_cap(cap), "cap")
            q = torch.randn(nh * hd, device="cuda", generator=g)
            K.attn_decode(q, kc, vc, torch.tensor([pos], dtype=torch.int32, device="cuda"), hd ** -0.5, part, tickets, out)
            want = R.attention(q.view(1, nh, hd), kc[:, :pos + 1].transpose(0, 1), vc[:, :pos + 1].transpose(0, 1),
                               pos).reshape(-1)
            assert not K.attn_error(tickets), turn
            assert bool(((out.float() - want).abs() <= 2 * size * (1 + want.abs()) / math.sqrt(1 + pos / 64)).all()), turn
    finally:
        K.check(K.kernels().cake_attn_set_split_cap(0), "cap")
        K.attn_set_single_max(prev)


@pytest.mark.parametrize("first,then", [(4, 2), (4, 1), (8, 2), (2, 4), (1, 8)])
@pytest.mark.parametrize("hd", [64, 128])
def test_groups_of_two_sizes_share_a_workspace(cuda, first, then, hd):
    """Launches of any group tag by one count: splits of the launch before, whose group was another, are not this one's.
    Dropped ones end in the error word, whatever the workspace holds."""
    nkv, S, pos = 2, 2048, 1500
    g = torch.Generator(device="cuda").manual_seed(hd)
    kc = torch.randn(nkv, S, hd, device="cuda", generator=g).bfloat16()
    vc = torch.randn(nkv, S, hd, device="cuda", generator=g).bfloat16()
    p = torch.tensor([pos], dtype=torch.int32, device="cuda")
    part = torch.zeros(K.attn_workspace_numel(nkv * max(first, then), hd, S), device="cuda")
    tickets = torch.zeros(2 * nkv + 2, dtype=torch.int32, device="cuda")

    def launch(n_rep):
        nh = n_rep * nkv
        q, out = torch.randn(nh * hd, device="cuda", generator=g), torch.empty(nh * hd, device="cuda", dtype=torch.bfloat16)
        K.attn_decode(q, kc, vc, p, hd ** -0.5, part, tickets, out)
        want = R.attention(q.view(1, nh, hd), kc[:, :pos + 1].transpose(0, 1), vc[:, :pos + 1].transpose(0, 1), pos)
        return bool(((out.float() - want.reshape(-1)).abs() <= 2.0 ** -6 * (1 + want.reshape(-1).abs()) / math.sqrt(1 + pos / 64)).all())
    for n_rep in (first, then, first, first, then):
        assert launch(n_rep) and not K.attn_error(tickets)
    K.attn_clear_error(tickets)
    launch(first)
    K.attn_debug_drop_partials(True)
    try:
        launch(then)
        torch.cuda.synchronize()
    finally:
        K.attn_debug_drop_partials(False)
    assert K.attn_error(tickets)


# groups whole, in parts and of one head; as many kv heads as take more splits in long contexts, and one more
@pytest.mark.parametrize("nh,nkv,hd", [(16, 2, 64), (64, 8, 128), (8, 2, 128), (8, 8, 64), (18, 9, 64)])
def test_long_contexts(cuda, nh, nkv, hd):
    """To either side of the length that takes twice the splits, in the graphs' caps and without; f32 attention within a
    rounding of 16-bit queries and result."""
    S, long = 28736, K._ATTN_LONG
    g = torch.Generator(device="cuda").manual_seed(nh)
    kc = torch.randn(nkv, S, hd, device="cuda", generator=g).bfloat16()
    vc = torch.randn(nkv, S, hd, device="cuda", generator=g).bfloat16()
    part = torch.zeros(K.attn_workspace_numel(nh, hd, S), device="cuda")
    tickets = torch.zeros(2 * nkv + 2, dtype=torch.int32, device="cuda")
    out = torch.empty(nh * hd, device="cuda", dtype=torch.bfloat16)
    assert K.attn_split_caps(S) == [8, 16, 32] and K.attn_splits(long) <= 16 < K.attn_splits(long + 1)
    for pos in (long - 1, long, S - 1, 700, long):
        for cap in (16, 32, 0):
            q = torch.randn(nh * hd, device="cuda", generator=g)
            with K.attn_split_cap(cap):
                K.attn_decode(q, kc, vc, torch.tensor([pos], dtype=torch.int32, device="cuda"), hd ** -0.5, part, tickets, out)
            want = R.attention(q.view(1, nh, hd), kc[:, :pos + 1].transpose(0, 1), vc[:, :pos + 1].transpose(0, 1), pos).reshape(-1)
            assert not K.attn_error(tickets)
            assert bool(((out.float() - want).abs() <= 2.0 ** -6 * (1 + want.abs()) / math.sqrt(1 + pos / 64)).all()), (pos, cap)
