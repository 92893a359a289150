"""16-bit projections of 17 to 64 rows (gemm_rows16.hip) against fp64: every number of row blocks and of tiles a workgroup, waves
without k-pairs and with odd numbers of them, ragged last workgroups; and which calls take the kernel."""
import pytest
import torch

from edgellm import ops
from edgellm.models.layers import Linear

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
    part = ops.ext().gemm_rows16(x, ops.pack_bf16_weight(w), b, N, 0, S=S)
    assert part.shape == (S, M, N)
    assert ((part.double().sum(0) - ref - b.double()).abs() <= 2 * K ** 0.5 * 2.0 ** -23 * (mag + b.double().abs()) + 1e-6).all()


def test_which_calls(cuda):
    """The kernel serves plain dense calls of an unwatched layer; the others keep the products they had."""
    x, w, b, ref, mag = _data(cuda, 20, 512, 512, torch.float16)
    assert ops.rows16_ok(x, w, b) and not ops.rows16_ok(x[:16], w, b) and not ops.rows16_ok(x.float(), w, b)
    assert not ops.rows16_ok(x.repeat(4, 1)[:65], w, b) and not ops.rows16_ok(x.t().contiguous().t(), w, b)
    flat = torch.empty(20 * 512 + 1, dtype=torch.float16, device=cuda)
    odd = flat[1:].view(20, 512).copy_(x)                   # two bytes off
    one = torch.ones(1, device=cuda, dtype=torch.float16)
    assert not ops.rows16_ok(odd, w, b) and not ops.rows16_ok(x, w, one)
    lin = Linear(512, 512, True, torch.float16, cuda)
    lin.weight.data.copy_(w)
    lin.bias.data.copy_(b)
    for v in (x, odd, x.view(4, 5, 512), x.t().contiguous().t(), x[:3], x.repeat(4, 1)):
        y, r = lin(v), torch.nn.functional.linear(v, w, b)
        assert y.shape == r.shape and (y.double() - r.double()).abs().max() <= 2.0 ** -9 * float(r.abs().max())
    add = torch.randn(512, device=cuda).half().expand(20, 512)    # strides of its own
    assert torch.equal(lin(x, add=add), lin(x) + add)
    g = x.clone().requires_grad_()
    lin(g).float().sum().backward()
    assert torch.allclose(g.grad.double(), w.double().sum(0).expand(20, -1), rtol=2e-3, atol=2e-3)
    with torch.no_grad():
        v = torch.func.vmap(lin)(x[None].expand(3, -1, -1))
        assert (v.double() - (ref + b.double())).abs().max() <= 2.0 ** -9 * float(ref.abs().max() + 4)
        seen = []
        plain = torch.nn.functional.linear(x, w, b)
        lin.register_forward_pre_hook(lambda m, a: seen.append(a[0]))
        assert torch.equal(lin(x), plain) and len(seen) == 1 and not lin.rows16_ok(x)


@pytest.mark.parametrize("M", [17, 32, 33, 45, 64])
@pytest.mark.parametrize("N,K", [(16, 128), (48, 1152), (4112, 384), (12304, 256), (16384, 640)])
def test_int8_rows(cuda, M, N, K):
    """Sums of int8 products are exact: the result is one chain of roundings."""
    g = torch.Generator(device=cuda).manual_seed(M + N + K)
    q = torch.randint(-127, 128, (M, K), generator=g, device=cuda, dtype=torch.int8)
    w = torch.randint(-127, 128, (N, K), generator=g, device=cuda, dtype=torch.int8)
    sa, sw = (torch.rand(n, generator=g, device=cuda) * 1e-2 + 1e-3 for n in (M, N))
    b = torch.randn(N, generator=g, device=cuda).bfloat16()
    y = ops.ext().w8a8_gemm(q, sa, ops.pack_int8_weight(w), sw, b, N, K)
    s = (q.double() @ w.double().T).float() * sa[:, None]
    ref = s.double() * sw.double() + b.double()
    assert ((y.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2.0 ** -22 * (s.abs() * sw)).all()


@pytest.mark.parametrize("over", [0, 1, 40])
@pytest.mark.parametrize("M,N,K", [(17, 2560, 2560), (45, 7680, 2560), (64, 48, 384), (33, 8208, 512)])
def test_llmint8_rows_with_their_outlier_columns(cuda, M, N, K, over):
    """One launch, bit for bit the product and the outlier columns' launch after it; activation and addend of that."""
    C, g = ops.ext(), torch.Generator(device=cuda).manual_seed(M + over)
    x = torch.randn(M, K, generator=g, device=cuda).clamp(-5, 5).bfloat16()
    at = torch.randperm(K, generator=g, device=cuda)[:over]
    x[torch.randint(0, M, (over,), generator=g, device=cuda), at] = 9.0
    w = torch.randint(-127, 128, (N, K), generator=g, device=cuda, dtype=torch.int8)
    scb, b = torch.rand(N, generator=g, device=cuda) + 0.5, torch.randn(N, generator=g, device=cuda).bfloat16()
    q, sa, cols, count = C.llmint8_prep_rows(x, 6.0)
    assert int(count) == over and cols[:over].tolist() == sorted(at.tolist())
    kept = x.float().clone()
    kept[:, at] = 0
    # (PyTorch divides by a number as a product with its rounded inverse: two roundings of 2^-24 apart)
    assert torch.allclose(sa, kept.abs().amax(1).clamp_min(1e-8) / 127, rtol=2.0 ** -22, atol=0) and not q[:, at].any()
    wp, wt, sw = ops.pack_int8_weight(w), w.t().contiguous(), scb / 127.0
    two = C.w8a8_gemm(q, sa, wp, sw, b, N, K)
    C.llmint8_outlier_rows(two, x, cols, count, wt, scb)
    one = C.llmint8_rows(q, sa, x, cols, count, wp, sw, b, wt, scb, N, 0, None)
    assert torch.equal(one, two)
    add = torch.randn(M, N, device=cuda).bfloat16()
    assert torch.equal(C.llmint8_rows(q, sa, x, cols, count, wp, sw, b, wt, scb, N, 0, add), two + add)
    for act, approx in ((1, "tanh"), (2, "none")):
        z = C.llmint8_rows(q, sa, x, cols, count, wp, sw, b, wt, scb, N, act, None).double()
        r = torch.nn.functional.gelu(two.double(), approximate=approx)
        assert ((z - r).abs() <= 2.0 ** -7 * r.abs() + 1e-6 * two.double().abs() + 1e-7).all()


@pytest.mark.parametrize("M,K", [(18, 96), (40, 2080), (513, 160), (1024, 64), (1025, 2080)])
def test_flags_of_few_and_many_rows(cuda, M, K):
    x = torch.randn(M, K, device=cuda).clamp(-5, 5).bfloat16()
    x[M - 1, K - 1], x[0, 3], x[M // 2, 31] = 7.0, -8.0, float("inf")
    q, sa, cols, count = ops.ext().llmint8_prep_rows(x, 6.0)
    assert cols[:int(count)].tolist() == sorted({3, 31, K - 1})
