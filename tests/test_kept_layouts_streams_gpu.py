"""Weight layouts that are formed on the first call and kept: the host waits for none of them, one that is formed while a graph is
recorded is the graph's alone, one that is not there yet when a graph that reads it is recorded is waited for, and copies are whole."""
import copy
import io

import pytest
import torch

from edgellm.models import build_model, tiny
from edgellm.models.layers import Linear
from edgellm.quant.linear import LLMInt8Linear

pytestmark = pytest.mark.gpu
KINDS = ["linear", "tied", "llm.int8"]


def _case(kind, cuda):
    """(module, a call that reads its layout, the call's result by a module of its own)."""
    g = torch.Generator(device=cuda).manual_seed(1)
    w = torch.randn(512, 256, device=cuda, generator=g).to(torch.bfloat16)
    x = torch.randn(1, 256, device=cuda, generator=g).to(torch.bfloat16)

    def make():
        if kind == "tied":
            m = build_model(tiny("llama", num_layers=1), dtype=torch.bfloat16, device=cuda, seed=3)
            h = x[:, :m.embed.shape[1]].contiguous()
            return m, lambda n=m: n._tied_head(h)
        lin = Linear(256, 512, dtype=torch.bfloat16, device=cuda)
        lin.weight.copy_(w)
        m = lin if kind == "linear" else LLMInt8Linear.from_float(lin)
        return m, lambda n=m: n(x)
    want = make()[1]()
    m, call = make()
    torch.cuda.synchronize()
    return m, call, want


def _busy(stream):
    """Some 60 ms of work queued on ``stream``; the event behind it."""
    with torch.cuda.stream(stream):
        a = torch.ones(4096, 4096, device="cuda:0", dtype=torch.bfloat16)
        for _ in range(500):
            a @ a
        return stream.record_event()


@pytest.mark.parametrize("kind", KINDS)
@torch.no_grad()
def test_first_call_does_not_wait(cuda, kind):
    _, call, want = _case(kind, cuda)
    one, two = torch.cuda.Stream(cuda), torch.cuda.Stream(cuda)
    behind = _busy(one)
    with torch.cuda.stream(one):
        first = call()
    assert not behind.query()
    with torch.cuda.stream(two):                             # waits on the card for the layout, not on the host
        second = call()
    assert not behind.query()
    torch.cuda.synchronize()
    assert torch.equal(first, want) and torch.equal(second, want) and torch.equal(call(), want)


@pytest.mark.parametrize("kind", KINDS)
@torch.no_grad()
def test_layout_formed_in_a_graph_stays_there(cuda, kind):
    _, call, want = _case(kind, cuda)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = call()
    assert torch.equal(call(), want)                         # (before the graph has run at all)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(call(), want)


@pytest.mark.parametrize("kind", KINDS)
@torch.no_grad()
def test_graph_recorded_while_the_layout_is_formed(cuda, kind):
    m, call, want = _case(kind, cuda)
    one, two = torch.cuda.Stream(cuda), torch.cuda.Stream(cuda)
    behind = _busy(one)
    with torch.cuda.stream(one):
        call()
    assert not behind.query()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(two):
        g.capture_begin()                                    # (torch.cuda.graph would wait for the device first)
        out = call()
        g.capture_end()
    assert behind.query()
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(call(), want)


@pytest.mark.parametrize("kind", KINDS)
@torch.no_grad()
def test_copies(cuda, kind):
    m, call, want = _case(kind, cuda)
    one = torch.cuda.Stream(cuda)
    _busy(one)
    with torch.cuda.stream(one):
        call()
    if kind != "tied":                                       # (a whole model is saved by its checkpoint)
        f = io.BytesIO()
        torch.save(m, f)
        f.seek(0)
        assert torch.equal(call(torch.load(f, weights_only=False)), want)
    assert torch.equal(call(copy.deepcopy(m)), want)
