"""Weight layouts that are built on the first call and kept: another stream may read them as soon as they are there."""
import pytest
import torch

from edgellm import ops
from edgellm.models import build_model, tiny
from edgellm.models.layers import Linear
from edgellm.quant.linear import LLMInt8Linear

pytestmark = pytest.mark.gpu


def _busy(stream):
    """About 20 ms of work queued on ``stream``, so that what follows there is not done when the host returns."""
    with torch.cuda.stream(stream):
        a = torch.ones(4096, 4096, device="cuda:0", dtype=torch.bfloat16)
        for _ in range(60):
            a @ a


@pytest.mark.parametrize("kind", ["linear", "tied", "llm.int8"])
def test_layout_read_from_another_stream(cuda, kind):
    one, two = torch.cuda.Stream(cuda), torch.cuda.Stream(cuda)
    g = torch.Generator(device=cuda).manual_seed(1)
    w = torch.randn(512, 256, device=cuda, generator=g).to(torch.bfloat16)
    x = torch.randn(4, 256, device=cuda, generator=g).to(torch.bfloat16)
    if kind == "linear":
        m = Linear(256, 512, dtype=torch.bfloat16, device=cuda)
        m.weight.copy_(w)
        build, want = (lambda: m.decode_weight(x)), ops.pack_bf16_weight(w)
    elif kind == "tied":
        m = build_model(tiny("llama", num_layers=1), dtype=torch.bfloat16, device=cuda, seed=3)
        h = x[:, :m.embed.shape[1]].contiguous()
        build, want = (lambda: (m._tied_head(h), m._embed_wp)[1]), ops.pack_bf16_weight(m.embed.detach())
    else:
        lin = Linear(256, 512, dtype=torch.bfloat16, device=cuda)
        lin.weight.copy_(w)
        m = LLMInt8Linear.from_float(lin)
        m._weight_t = None
        build, want = (lambda: m._transposed(cuda) or m._weight_t), m.weight_i8.t().contiguous()
    torch.cuda.synchronize()
    _busy(one)
    with torch.cuda.stream(one):
        build()
    with torch.cuda.stream(two):
        got = build().clone()
    two.synchronize()
    assert torch.equal(got, want)
