"""Calls whose ops are recorded, rewritten or watched keep PyTorch ops; only the others reach kernels that read memory."""
import ctypes

import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode
from torch.utils.flop_counter import FlopCounterMode

import edgellm  # noqa: F401
from edgellm import ops


class _Raw:
    """The extension's fp32 product, its result written past PyTorch."""

    calls = 0

    def gemv_f32(self, x, w, bias):
        self.calls += 1
        y = torch.empty(*x.shape[:-1], w.shape[0])
        ref = (x.detach().double() @ w.detach().double().t()).float().contiguous()
        ctypes.memmove(y.data_ptr(), ref.data_ptr(), ref.numel() * 4)
        return y


@pytest.fixture
def raw(monkeypatch):
    r = _Raw()
    monkeypatch.setattr(ops, "_gpu", lambda t: True)
    monkeypatch.setattr(ops, "available", lambda: True)
    monkeypatch.setattr(ops, "ext", lambda: r)
    monkeypatch.setattr(ops, "bf16_decode_mode", lambda *a, **k: 0)
    return r


def _xw(seed=0):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(2, 64, generator=g), torch.randn(32, 64, generator=g)


@pytest.mark.parametrize("kw", [{}, {"pre_dispatch": True}, {"tracing_mode": "fake"}, {"tracing_mode": "symbolic"}])
def test_make_fx_records_the_product(raw, kw):
    x, w = _xw()
    graph = make_fx(lambda a, b: ops.linear_bf16(a, b), **kw)(x, w)
    x2, w2 = _xw(1)
    assert raw.calls == 0 and torch.allclose(graph(x2, w2), torch.nn.functional.linear(x2, w2), atol=1e-4)


def test_jit_trace_records_the_product(raw):
    x, w = _xw()
    traced = torch.jit.trace(lambda a, b: ops.linear_bf16(a, b), (x, w), check_trace=False)
    x2, w2 = _xw(1)
    assert raw.calls == 0 and torch.allclose(traced(x2, w2), torch.nn.functional.linear(x2, w2), atol=1e-4)


def test_modes_and_transforms_keep_the_library_product(raw):
    x, w = _xw()
    ref = torch.nn.functional.linear(x, w)
    with FlopCounterMode(display=False) as flops:
        ops.linear_bf16(x, w)
    assert flops.get_total_flops() == 2 * 2 * 64 * 32

    class Seen(TorchFunctionMode):
        linear = 0

        def __torch_function__(self, f, types, args=(), kwargs=None):
            self.linear += f is torch.nn.functional.linear or f is torch._C._nn.linear
            return f(*args, **(kwargs or {}))

    with Seen() as seen:
        ops.linear_bf16(x, w)
    assert seen.linear
    assert torch.allclose(torch.func.functionalize(ops.linear_bf16)(x, w), ref, atol=1e-4)
    assert torch.allclose(torch.func.vmap(lambda r: ops.linear_bf16(r, w))(x), ref, atol=1e-4)
    assert torch.allclose(ops.linear_bf16(torch._neg_view(x), w), -ref, atol=1e-4)
    assert torch.allclose(ops.linear_bf16(x, w.to_sparse_csr()), ref, atol=1e-4)
    y = ops.linear_bf16(x.clone().requires_grad_(), w)
    assert y.requires_grad and raw.calls == 0


def test_a_plain_call_reaches_the_kernel(raw):
    x, w = _xw()
    assert torch.allclose(ops.linear_bf16(x, w), torch.nn.functional.linear(x, w), atol=1e-4)
    with torch.no_grad():
        ops.linear_bf16(x, torch.nn.Parameter(w))
    with torch.inference_mode():
        ops.linear_bf16(x, w)
    assert raw.calls == 3


def test_a_bias_that_broadcasts_is_the_librarys(raw):
    x, w = _xw()
    col, w2 = torch.tensor([[1.0], [2.0]]), w[:2].contiguous()
    assert torch.allclose(ops.linear_bf16(x, w2, col), x @ w2.t() + col, atol=1e-4)
    with pytest.raises(RuntimeError):
        ops.linear_bf16(x[:1].expand(3, 64).contiguous(), w2, col)
    assert raw.calls == 0


@pytest.mark.gpu
def test_llmint8_added_row_keeps_its_gradient_and_transforms():
    """One row, the sum where autograd, forward mode, vmap and dispatch modes see it: add's own gradient, tangent and batch."""
    from edgellm.models.layers import Linear
    from edgellm.quant import LLMInt8Linear
    lin = Linear(128, 96, bias=False, device="cuda:0")
    lin.weight.data.copy_(torch.randn(96, 128) * 0.05)
    m = LLMInt8Linear.from_float(lin)
    x, add = torch.randn(1, 128).bfloat16().cuda(), torch.randn(1, 96).bfloat16().cuda()
    with torch.no_grad():
        ref = m(x, add=add)                                # in the epilogue
    leaf, up = add.clone().requires_grad_(), torch.randn(1, 96).bfloat16().cuda()
    y = m(x, add=leaf)
    (grad,) = torch.autograd.grad(y + leaf, leaf, up)      # add reaches the result another way as well
    assert torch.equal(y, ref) and torch.equal(grad, 2 * up)
    with torch.autograd.forward_ad.dual_level():
        dual = m(x, add=torch.autograd.forward_ad.make_dual(add, up))
        assert torch.equal(torch.autograd.forward_ad.unpack_dual(dual).tangent, up)
    rows = torch.stack([add, add * 2])
    assert torch.equal(torch.func.vmap(lambda a: m(x, add=a))(rows), torch.stack([ref, m(x) + add * 2]))
    with FlopCounterMode(display=False):
        assert torch.equal(m(x, add=add), ref)


def test_a_row_joins_an_epilogue_only_as_plain_memory():
    from edgellm.quant.linear import _epilogue_row
    x, add = torch.zeros(1, 8, dtype=torch.bfloat16), torch.zeros(1, 8, dtype=torch.bfloat16)
    leaf = add.clone().requires_grad_()
    assert _epilogue_row(add, x) and not _epilogue_row(leaf, x) and not _epilogue_row(add.float(), x)
    assert not _epilogue_row(torch.zeros(1, 16, dtype=torch.bfloat16)[:, ::2], x)
    with torch.no_grad():
        assert _epilogue_row(leaf, x)
    seen = []
    torch.func.vmap(lambda a: (seen.append(_epilogue_row(a, x)), a * 1)[1])(add)
    torch.func.jvp(lambda a: (seen.append(_epilogue_row(a, x)), a * 1)[1], (add,), (add,))
    make_fx(lambda a: (seen.append(_epilogue_row(a, x)), a * 1)[1])(add)
    assert seen == [False] * 3
