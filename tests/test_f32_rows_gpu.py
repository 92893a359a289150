"""A few fp32 rows through gemv_f32.hip against 64-bit sums, at the edges of its row groups, k chunks and waves; calls it does
not take keep the library's product."""
import pytest
import torch

from edgellm import ops

pytestmark = pytest.mark.gpu


def _operands(M, N, K, seed=0):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(*s, generator=g).cuda() for s in ((M, K), (N, K), (N,))]


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("N,K", [(1, 4), (3, 252), (4, 256), (5, 260), (33, 1024), (1023, 1028), (1024, 4096), (1025, 4096),
                                 (4097, 516), (8192, 768)])
def test_f32_rows(M, N, K):
    x, w, b = _operands(M, N, K, M)
    assert ops.f32_rows_ok(x, w, b) == (M <= 4 or N * K <= 1 << 22)
    for bias in (None, b):
        got = ops.linear_bf16(x, w, bias).double().cpu()
        ref = x.double().cpu() @ w.double().cpu().t() + (0 if bias is None else bias.double().cpu())
        # a lane chains at most K / 64 + 4 fused products, then come 6 + 4 sums of sums: each step rounds by 2^-24 of what
        # it holds, which the sum of sizes bounds
        size = x.double().cpu().abs() @ w.double().cpu().abs().t() + 10
        assert ((got - ref).abs() <= (16 + K / 64) * 2.0 ** -24 * size).all()


def test_f32_rows_nan_and_inf_stay_in_their_column():
    x, w, _ = _operands(2, 20, 260)
    w[7, 259], w[9, 0] = float("nan"), float("inf")
    y = ops.linear_bf16(x, w)
    bad = torch.zeros(20, dtype=torch.bool)
    bad[7] = bad[9] = True
    assert torch.equal(~y.isfinite().all(0).cpu(), bad) and y[:, 9].isinf().all()


def test_f32_rows_leaves_other_calls_to_the_library():
    x, w, b = _operands(2, 64, 256)
    ref = torch.nn.functional.linear(x, w, b)
    assert not ops.f32_rows_ok(torch.cat([x] * 5), w) and not ops.f32_rows_ok(x, w.t().contiguous().t())
    assert not ops.f32_rows_ok(torch.randn(2, 257, device="cuda")[:, 1:], w)
    xr = x.clone().requires_grad_()
    y = ops.linear_bf16(xr, w, b)
    y.sum().backward()
    assert torch.allclose(xr.grad, w.sum(0).expand(2, -1), atol=1e-4)
    batched = torch.func.vmap(lambda r: ops.linear_bf16(r, w, b))(x)
    _, tangent = torch.func.jvp(lambda r: ops.linear_bf16(r, w, b), (x,), (x,))
    with torch.autograd.forward_ad.dual_level():
        dual = ops.linear_bf16(torch.autograd.forward_ad.make_dual(x, x), w, b)
        assert torch.allclose(torch.autograd.forward_ad.unpack_dual(dual).tangent, ref - b, atol=1e-4)
    with torch.autocast("cuda", torch.bfloat16):
        assert ops.linear_bf16(x, w, b).dtype == torch.bfloat16
    assert torch.allclose(batched, ref, atol=1e-4) and torch.allclose(tangent, ref - b, atol=1e-4)
