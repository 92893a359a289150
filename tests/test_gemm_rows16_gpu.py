"""16-bit projections of 17 to 64 rows (gemm_rows16.hip) against fp64: every number of row blocks and of tiles a workgroup, waves
without k-pairs and with odd numbers of them, ragged last workgroups; and which calls take the kernel."""
import pytest
import torch

from edgellm import ops

pytestmark = pytest.mark.gpu


def _check(y, ref, mag, K, dtype):
    """Rounding of the result (and of gate and up before it), and K fp32 sums of products whose magnitudes add up to ``mag``."""
    eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    assert ((y.double() - ref).abs() <= 4 * eps * ref.abs() + 2 * K ** 0.5 * 2.0 ** -23 * mag + 1e-6).all()


def _data(cuda, M, N, K, dtype):
    g = torch.Generator(device=cuda).manual_seed(M * 31 + N + K)
    x = torch.randn(M, K, generator=g, device=cuda).to(dtype)
    w = (torch.randn(N, K, generator=g, device=cuda) * K ** -0.5).to(dtype)
    b = torch.randn(N, generator=g, device=cuda).to(dtype)
    return x, w, b, x.double() @ w.double().T, x.double().abs() @ w.double().abs().T


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [17, 32, 33, 49, 64])
@pytest.mark.parametrize("N,K", [(16, 64), (48, 576), (4112, 1088), (8208, 192), (12304, 512), (16384, 640)])
def test_plain_gelu_and_addend(cuda, M, N, K, dtype):
    x, w, b, ref, mag = _data(cuda, M, N, K, dtype)
    wp, C = ops.pack_bf16_weight(w), ops.ext()
    y = C.gemm_rows16(x, wp, b, N, 0)
    _check(y, ref + b.double(), mag + b.double().abs(), K, dtype)
    add = torch.randn(M, N, device=cuda).to(dtype)
    assert torch.equal(C.gemm_rows16(x, wp, b, N, 0, add), y + add)
    for epi, approx in ((2, "tanh"), (3, "none")):
        z = C.gemm_rows16(x, wp, None, N, epi)
        p = C.gemm_rows16(x, wp, None, N, 0).double()       # gelu of the rounded output
        r = torch.nn.functional.gelu(p, approximate=approx)
        _check(z, r, p.abs(), 1, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,F", [(17, 16), (32, 4112), (33, 8208), (48, 12272), (64, 48), (64, 8192), (20, 12304)])
def test_swiglu(cuda, M, F, dtype):
    x, w, b, ref, mag = _data(cuda, M, 2 * F, 320, dtype)
    y = ops.ext().gemm_rows16(x, ops.pack_bf16_weight(w), b, 2 * F, 1)
    g, u = (ref + b.double()).chunk(2, -1)
    eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    gr, ur = g.to(dtype).double(), u.to(dtype).double()
    tol = 4 * eps * (torch.nn.functional.silu(gr) * ur).abs() + 2.2 * eps * g.abs() * u.abs() + 1e-4
    assert ((y.double() - torch.nn.functional.silu(gr) * ur).abs() <= tol).all()


@pytest.mark.parametrize("M", [17, 40, 64])
@pytest.mark.parametrize("N,K,S", [(1024, 1024, 4), (2064, 1600, 4), (4096, 2048, 4), (6160, 576, 2), (9216, 512, 2)])
def test_slices(cuda, M, N, K, S):
    x, w, b, ref, mag = _data(cuda, M, N, K, torch.bfloat16)
    part = ops.ext().gemm_bf16_ring(x, ops.pack_bf16_weight(w), b, N, 3, S)
    assert part.shape == (S, M, N)
    assert ((part.double().sum(0) - ref - b.double()).abs() <= 2 * K ** 0.5 * 2.0 ** -23 * (mag + b.double().abs()) + 1e-6).all()


def test_which_calls(cuda):
    """The kernel serves plain dense calls with a kept packed weight; PyTorch's own product serves the others, as before."""
    x, w, b, ref, mag = _data(cuda, 20, 512, 512, torch.float16)
    wp = ops.pack_bf16_weight(w)
    assert ops.rows16_ok(x, w, b) and not ops.rows16_ok(x[:16], w, b) and not ops.rows16_ok(x.float(), w, b)
    assert not ops.rows16_ok(x.repeat(4, 1)[:65], w, b) and not ops.rows16_ok(x.t().contiguous().t(), w, b)
    flat = torch.empty(20 * 512 + 1, dtype=torch.float16, device=cuda)
    odd = flat[1:].view(20, 512).copy_(x)                   # two bytes off
    assert not ops.rows16_ok(odd, w, b)
    one = torch.ones(1, device=cuda, dtype=torch.float16)
    for args in ((x, w, b), (odd, w, b), (x, w, one), (x.view(4, 5, 512), w, None), (x.t().contiguous().t(), w, b)):
        y = ops.linear_bf16(*args, packed=wp)
        r = torch.nn.functional.linear(*args)
        assert y.shape == r.shape and (y.double() - r.double()).abs().max() <= 2.0 ** -9 * float(r.abs().max())
    lone = torch.randn(512, device=cuda).half()             # an addend that broadcasts
    assert torch.equal(ops.linear_bf16(x, w, b, packed=wp, add=lone), ops.linear_bf16(x, w, b, packed=wp) + lone)
    g = x.clone().requires_grad_()
    ops.linear_bf16(g, w, b, packed=wp).float().sum().backward()
    assert torch.allclose(g.grad.double(), w.double().sum(0).expand(20, -1), rtol=2e-3, atol=2e-3)
    with torch.no_grad():
        v = torch.func.vmap(lambda r: ops.linear_bf16(r, w, b, packed=wp))(x[None].expand(3, -1, -1))
    assert (v.double() - (ref + b.double())).abs().max() <= 2.0 ** -9 * float(ref.abs().max() + 4)
