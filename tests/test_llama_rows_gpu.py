"""A run of Llama blocks as one native call against the separate calls it replaces: the same
kernels in the same order, so the same bits."""
import pytest
import torch

from cake_amd.models.llama3.blocks import LayerStack
from cake_amd.models.llama3.config import LlamaConfig
from cake_amd.models.llama3.weights import BlockWeights

pytestmark = pytest.mark.gpu


def _stack(dt, H=512, I=1024, nh=4, nkv=2, layers=3, max_seq=512):
    cfg = LlamaConfig(hidden_size=H, intermediate_size=I, vocab_size=64, num_hidden_layers=layers,
                      num_attention_heads=nh, num_key_value_heads=nkv)
    g = torch.Generator(device="cuda").manual_seed(5)

    def t(*shape):
        s = shape[-1] ** -0.5 if len(shape) == 2 else 1.0
        return (torch.randn(*shape, device="cuda", generator=g) * s).to(dt)
    hd = cfg.head_dim
    w = {i: BlockWeights(ln1=t(H), wq=t(nh * hd, H), wk=t(nkv * hd, H), wv=t(nkv * hd, H),
                         wo=t(H, nh * hd), ln2=t(H), wg=t(I, H), wu=t(I, H), wd=t(H, I))
         for i in range(layers)}
    return LayerStack(cfg, w, "cuda", dt, max_seq, "hip")


def _separate(stack, hidden, layers, pos0, session):
    kv = stack.cache(session)
    for li in layers:
        s = stack.slot_of[li]
        stack._prefill_hip(hidden, stack.weights[li], kv.k[s], kv.v[s], pos0)
    return hidden


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("T,pos0", [(2, 0), (5, 9), (33, 0), (64, 100), (65, 0), (300, 212)])
def test_same_bits(dt, T, pos0):
    stack = _stack(dt)
    layers = [0, 2, 1]   # any order of any of them
    h = torch.randn(T, 512, device="cuda")
    for s in (1, 2):     # what lies before the rows
        kv = stack.cache(s)
        g = torch.Generator(device="cuda").manual_seed(3)
        for c in (kv.k, kv.v):
            c.copy_(torch.randn(c.shape, device="cuda", generator=g))
    want = _separate(stack, h.clone(), layers, pos0, 1)
    got = stack.forward(h.clone(), layers, pos0, 2)
    assert torch.equal(got, want) and bool(torch.isfinite(got).all())
    assert torch.equal(stack.cache(1).k, stack.cache(2).k)
    assert torch.equal(stack.cache(1).v, stack.cache(2).v)
    assert stack.cache(2).length == pos0 + T


def test_other_forms_take_the_separate_calls():
    """Head sizes and weights outside the native call's forms run as before."""
    from cake_amd.ops.llama_rows import block_rows
    stack = _stack(torch.bfloat16, H=96, I=160, nh=8, nkv=8)   # heads of 12
    kv, h = stack.cache(0), torch.randn(6, 96, device="cuda")
    args = ([stack.weights[0]], [0], kv.k, kv.v, stack.inv_freq, stack.cfg, 0, stack.scale)
    assert not block_rows(h, *args)
    stack = _stack(torch.bfloat16)
    kv, h = stack.cache(0), torch.randn(6, 512, device="cuda")
    wide = torch.zeros(512, 1032, device="cuda", dtype=torch.bfloat16)
    want = stack.forward(h.clone(), [0], 0)
    stack.weights[0].wd = wide[:, :1024].copy_(stack.weights[0].wd)   # rows 1032 apart
    assert not block_rows(h, [stack.weights[0]], [0], kv.k, kv.v, stack.inv_freq, stack.cfg, 0,
                          stack.scale)
    assert torch.equal(stack.forward(h.clone(), [0], 0), want)


@pytest.mark.parametrize("T", [20, 200])
def test_captured(T):
    stack = _stack(torch.bfloat16)
    x = torch.randn(3, T, 512, device="cuda")
    h = x[0].clone()
    stack.forward(h, [0, 1, 2], 0)   # buffers and plans before the capture
    graph, buf = torch.cuda.CUDAGraph(), x[0].clone()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        stack.forward(buf, [0, 1, 2], 0)
    for i in (1, 2, 0):
        buf.copy_(x[i])
        graph.replay()
        torch.cuda.synchronize()
        want = stack.forward(x[i].clone(), [0, 1, 2], 0)
        # few rows take other kernels under capture: rounding of 16-bit activations, 3 blocks
        assert float((buf - want).norm() / want.norm()) < 3 * 2 ** -8
