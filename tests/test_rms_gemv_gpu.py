"""Few bf16 rows normed and projected in one launch (rms_gemv.hip) against 64 bits: widths at the edges of its unrolled forms, rows up to
16, one tile and many, row strides; and the calls that stay two launches."""
import pytest
import torch

import edgellm.ops.seqmix as S
from edgellm.models.layers import Linear

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,K,N,extra,dt,one", [
    (1, 64, 16, 0, torch.bfloat16, True), (4, 384, 1536, 160, torch.bfloat16, True), (16, 512, 48, 8, torch.bfloat16, True),
    (3, 128, 32, 24, torch.bfloat16, True), (5, 192, 64, 0, torch.bfloat16, True), (2, 256, 160, 8, torch.bfloat16, True),
    (17, 384, 64, 0, torch.bfloat16, False), (2, 576, 64, 0, torch.bfloat16, False), (2, 96, 64, 0, torch.bfloat16, False),
    (2, 128, 24, 0, torch.bfloat16, False), (2, 128, 64, 4, torch.bfloat16, False), (2, 128, 64, 0, torch.float32, False)])
@torch.no_grad()
def test_against_64_bits(T, K, N, extra, dt, one):
    g = torch.Generator(device="cuda").manual_seed(K + N + T)
    u = (torch.randn(T, K + extra, device="cuda", generator=g) * 3).to(dt)
    w = 1 + 0.2 * torch.randn(K, device="cuda", generator=g)
    lin = Linear(K, N, False, dt, "cuda")
    lin.weight.copy_((torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).to(dt))
    calls = []
    ext, real = S._ext(), S._ext().sm_rms_gemv
    try:
        ext.sm_rms_gemv = lambda *a: calls.append(real(*a)) or calls[-1]
        got = S.rms_norm_linear(u, w, 1e-6, lin)
    finally:
        ext.sm_rms_gemv = real
    assert (bool(calls) and calls[-1] is not None) == one
    x = u[:, :K].double()
    x = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()
    ref, size = x @ lin.weight.double().t(), x.abs() @ lin.weight.double().abs().t()
    # the normed numbers are rounded to dt once and so is the result: half a unit in the last place each, fp32 sums besides
    half = 2.0 ** -9 if dt == torch.bfloat16 else 2.0 ** -24
    assert got.shape == (T, N) and got.dtype == dt
    assert ((got.double() - ref).abs() <= half * 1.01 * (size + ref.abs()) + K * 2.0 ** -24 * size).all()
