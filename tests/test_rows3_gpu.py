"""Three projections of the same few rows in one launch (gemv_f32.hip, decode_pair.hip) against float64 and, in fp32, bit for bit
against the single launches: widths beside a wave's 256 k and four rows, unequal sizes, every count of rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("sizes", [((1024, 4096), (1024, 1024), (1024, 1024)), ((5, 4), (1, 260), (130, 1020)), ((2048, 8192), (16, 64), (3, 2052))])
def test_fp32(cuda, M, sizes):
    from edgellm import ops
    g = torch.Generator().manual_seed(M)
    xs = [torch.randn(M, K, generator=g).cuda() for _, K in sizes]
    ws = [(torch.randn(N, K, generator=g) * K ** -0.5).cuda() for N, K in sizes]
    ys = ops.ext().gemv_rows3(xs[0], ws[0], xs[1], ws[1], xs[2], ws[2], *(N for N, _ in sizes))
    for y, x, w in zip(ys, xs, ws):
        assert torch.equal(y, ops.ext().gemv_f32(x, w, None))
        ref = x.double() @ w.double().t()
        assert ((y.double() - ref).abs() <= 2.0 ** -24 * x.shape[1] * (x.double().abs() @ w.double().abs().t()) + 1e-7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 2, 4])
@pytest.mark.parametrize("sizes", [((1024, 4096), (1024, 1024), (1024, 1024)), ((16, 64), (32, 320), (272, 2112))])
def test_16_bits(cuda, dtype, M, sizes):
    from edgellm import ops
    g = torch.Generator().manual_seed(M)
    xs = [torch.randn(M, K, generator=g).to(dtype).cuda() for _, K in sizes]
    ws = [(torch.randn(N, K, generator=g) * K ** -0.5).to(dtype).cuda() for N, K in sizes]
    p = [ops.pack_bf16_weight(w) for w in ws]
    ys = ops.ext().gemv_rows3(xs[0], p[0], xs[1], p[1], xs[2], p[2], *(N for N, _ in sizes))
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for y, x, w in zip(ys, xs, ws):
        ref = x.double() @ w.double().t()
        assert ((y.double() - ref).abs() <= eps * ref.abs() + 2.0 ** -24 * x.shape[1] * (x.double().abs() @ w.double().abs().t())).all()
