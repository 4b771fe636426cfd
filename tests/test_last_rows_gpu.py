"""Blocks of which only the last rows are read: the same rows, keys and values as of all of them."""
import hybrid_cases
import latent_cases
import pytest
import torch

from test_llama_rows_gpu import _stack

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("T,pos0,tail", [(64, 0, 1), (65, 0, 1), (66, 100, 3), (80, 5, 20), (80, 0, 21),
                                         (300, 0, 1), (300, 200, 70), (70, 0, 70)])
def test_last_rows(dt, T, pos0, tail):
    stack = _stack(dt)
    h = torch.randn(T, 512, device="cuda", generator=torch.Generator("cuda").manual_seed(T))
    g = torch.Generator(device="cuda").manual_seed(3)
    for c in (stack.cache(1).k, stack.cache(1).v):   # what lies before the rows
        c.copy_(torch.randn(c.shape, device="cuda", generator=g))
    stack.cache(2).k.copy_(stack.cache(1).k)
    stack.cache(2).v.copy_(stack.cache(1).v)
    want = stack.forward(h.clone(), [0, 1, 2], pos0, 1)[-tail:]
    got = stack.forward(h.clone(), [0, 1, 2], pos0, 2, tail=tail)[-tail:]
    # one block's products in other orders of sums: a 16-bit rounding apart here and there
    half = 2.0 ** (-8 if dt == torch.bfloat16 else -11)
    assert float((got - want).norm() / want.norm()) < half
    for a, b in ((stack.cache(1).k, stack.cache(2).k), (stack.cache(1).v, stack.cache(2).v)):
        assert torch.equal(a[:2], b[:2])   # the blocks before the last
        assert torch.equal(a[:, :, :pos0], b[:, :, :pos0]) and torch.equal(a[:, :, pos0 + T:], b[:, :, pos0 + T:])
        assert float((a.float() - b.float()).norm() / a.float().norm()) < half
    assert stack.cache(2).length == pos0 + T


HYBRID = [(hybrid_cases, n) for n in hybrid_cases.CASES] + [(latent_cases, n) for n in latent_cases.CASES]


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("cases,name", HYBRID, ids=lambda v: v if isinstance(v, str) else "")
def test_last_run_of_a_step(dt, cases, name):
    """Prompts of several lengths side by side, a wanted row amid one of them, one without any; then a
    token of each: against the same model with all rows in every run (which an observer asks for)."""
    from cake_amd.models.base import StepEntry
    from cake_amd.models.hybrid.model import HybridModel
    cfg, get, _ = cases.weights_of(cases.CASES[name])
    V = cfg.vocab_size
    lens = [70, 3, 40, 25]
    toks = [hybrid_cases.tokens(n + 1, V, seed=n) for n in lens]
    wants = [[69], [2], [12], []]
    got, ran = [], []
    for observe in (None, lambda x: None):
        model = HybridModel.build(cfg, get, "cuda", dt, 128, slots=6)
        whole = model._last_rows
        model._last_rows = lambda *a: ran.append(observe) or whole(*a)
        ids = [model.open_sequence() for _ in lens]
        out = model.step([StepEntry(i, t[:-1], w) for i, t, w in zip(ids, toks, wants)], observe=observe)
        # a second prompt behind the first, of rows enough to be left out again
        more = hybrid_cases.tokens(50, V, seed=9)
        out += model.step([StepEntry(ids[1], more, [49]), StepEntry(ids[3], more[:20], [19])], observe=observe)
        out += model.step([StepEntry(i, [t[-1]], [0]) for i, t in zip(ids, toks)], observe=observe)
        got.append([t.float() for t in out])
    assert ran == [None, None]
    half = 2.0 ** (-8 if dt == torch.bfloat16 else -11)
    for a, b in zip(*got):
        assert a.shape == b.shape
        if b.numel():   # some roundings of 16-bit activations apart, in the last run and what reads its rows
            assert float((a - b).norm() / b.norm()) < 6 * half


def test_wanted_rows_that_keep_the_whole_run():
    """Two rows of one sequence, more of them than a quarter, none: every row goes through."""
    from cake_amd.models.base import StepEntry
    from cake_amd.models.hybrid.model import HybridModel
    cfg, get, _ = hybrid_cases.weights_of(hybrid_cases.CASES["mixed"])
    model = HybridModel.build(cfg, get, "cuda", torch.bfloat16, 128, slots=24)
    model._last_rows = None
    t = hybrid_cases.tokens(80, cfg.vocab_size)
    for entries in ([(t, [78, 79])], [(t, [])], [(t[:3], [2])] * 22):
        ids = [model.open_sequence() for _ in entries]
        out = model.step([StepEntry(i, e, w) for i, (e, w) in zip(ids, entries)])
        assert [len(o) for o in out] == [len(w) for _, w in entries]
        for i in ids:
            model.close_sequence(i)
