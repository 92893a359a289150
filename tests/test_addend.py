"""The addend of a 16-bit projection joins the kernel's launch only as a dense tensor beside the rows; any other stays an op of PyTorch's,
which raises where it always did."""
import pytest
import torch

from edgellm import ops
from edgellm.models.layers import Linear


class _Ext:
    """Stands in for the kernels: keeps the addend that reached them."""
    def __init__(self):
        self.addends = []

    def gemm_rows16(self, x, packed, bias, N, epi, addend=None):
        self.addends.append(addend)
        return torch.zeros(*x.shape[:-1], N, dtype=x.dtype)

    def gemv_bf16(self, x, packed, bias, N, epi, addend=None):
        return self.gemm_rows16(x, packed, bias, N, epi, addend)


def test_an_addend_on_another_device_does_not_reach_the_rows_kernel(monkeypatch):
    ext = _Ext()
    monkeypatch.setattr(ops, "ext", lambda: ext)
    monkeypatch.setattr(ops, "raw_call", lambda *ts: True)
    x = torch.zeros(20, 64, dtype=torch.bfloat16)
    add = torch.zeros(20, 32, dtype=torch.bfloat16)
    ops.rows16(x, None, None, 32, None, add)
    try:
        ops.rows16(x, None, None, 32, None, add.to("meta"))
    except RuntimeError:
        pass                                                 # (the sum's own refusal, where it refuses)
    assert ext.addends[0] is add and ext.addends[1] is None


@pytest.mark.parametrize("kind", ["strides", "gradient"])
def test_what_is_no_dense_number_does_not_reach_the_gemv(monkeypatch, kind):
    ext = _Ext()
    monkeypatch.setattr(ops, "ext", lambda: ext)
    monkeypatch.setattr(ops, "bf16_decode_mode", lambda *a, **k: 1)
    x, w = torch.zeros(3, 64, dtype=torch.bfloat16), torch.zeros(32, 64, dtype=torch.bfloat16)
    add = torch.arange(32).bfloat16().expand(3, 32) if kind == "strides" else torch.ones(3, 32, dtype=torch.bfloat16, requires_grad=True)
    y = ops.linear_bf16(x, w, packed=w, add=add)
    assert ext.addends == [None] and torch.equal(y, add) and y.requires_grad == add.requires_grad
    ops.linear_bf16(x, w, packed=w, add=add.detach().contiguous())
    assert ext.addends[1] is not None


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [3, 16, 20, 70])
def test_an_addend_with_strides_of_its_own(cuda, rows):
    lin = Linear(256, 512, False, torch.bfloat16, cuda)
    lin.weight.data.normal_()
    x = torch.randn(rows, 256, device=cuda).bfloat16()
    for add in (torch.randn(512, device=cuda).bfloat16().expand(rows, 512), torch.randn(rows, 1024, device=cuda).bfloat16()[:, :512]):
        with torch.no_grad():
            assert torch.equal(lin(x, add=add), lin(x) + add)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [3, 20, 70])
def test_an_addend_in_host_memory_is_refused(cuda, rows):
    lin = Linear(256, 512, False, torch.bfloat16, cuda)
    lin.weight.data.normal_()
    x, add = torch.randn(rows, 256, device=cuda).bfloat16(), torch.randn(rows, 512).bfloat16()
    with torch.no_grad():
        with pytest.raises(RuntimeError, match="device|is on|cpu"):
            lin(x, add=add)
        assert torch.equal(lin(x, add=add.to(cuda)), lin(x) + add.to(cuda))
