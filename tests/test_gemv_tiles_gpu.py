"""16-bit GEMV of up to 16 rows, one tile of a workgroup's at a time (gemv_bf16.h gemv_tiles_body), against float64."""
import pytest
import torch

from edgellm import ops

pytestmark = pytest.mark.gpu

EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _operands(cuda, dtype, M, N, K):
    g = torch.Generator(device=cuda).manual_seed(M * 1009 + N * 31 + K)
    r = lambda *s: torch.randn(*s, generator=g, device=cuda)  # noqa: E731
    return r(M, K).to(dtype), (r(N, K) * K ** -0.5).to(dtype), r(N).to(dtype), r(M, N).to(dtype)


def _near(y, ref, bound):
    err = (y.double() - ref).abs()
    assert bool((err <= bound).all()), float((err - bound).max())


# K: less than a wave's k-pair each, ragged rounds, several rounds; N: one tile, ragged tiles a workgroup, over 1024 tiles; 8192 x 4096 is two
# tiles a workgroup from 11 rows on
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("N,K", [(16, 64), (48, 1088), (1040, 2560), (16400, 192), (8192, 4096)])
def test_plain_split_and_addend(cuda, dtype, M, N, K):
    x, w, b, add = _operands(cuda, dtype, M, N, K)
    wp = ops.pack_bf16_weight(w)
    exact = x.double() @ w.double().t() + b.double()
    # fp32 products added in any order: each of K terms is rounded at most once a sum, sums are below sum |x w|
    part = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t() + b.double().abs())
    y = ops.ext().gemv_bf16(x, wp, b, N, 0, None)
    _near(y, exact, part + EPS[dtype] * exact.abs() + 1e-7)
    z = ops.ext().gemv_bf16(x, wp, b, N, 0, add)
    assert torch.equal(z, (y.float() + add.float()).to(dtype))
    for S in (1, 2, 5):
        if S <= K // 64:
            _near(ops.ext().gemv_bf16_splitk(x, wp, b, N, S).double().sum(0), exact, part)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 3, 4, 6, 16])
@pytest.mark.parametrize("N,K", [(32, 64), (1056, 1088), (16416, 192), (8192, 4096)])
@pytest.mark.parametrize("epi", [1, 2, 3])
def test_activations(cuda, dtype, M, N, K, epi):
    x, w, b, _ = _operands(cuda, dtype, M, N, K)
    y = ops.ext().gemv_bf16(x, ops.pack_bf16_weight(w), b, N, epi, None).double()
    u = x.double() @ w.double().t() + b.double()
    if epi == 1:
        ref = torch.nn.functional.silu(u[:, :N // 2]) * u[:, N // 2:]
        # the rounded gate and up, the rounded result: each moves it by its size or, where silu is flat, by |up| of the gate
        bound = EPS[dtype] * (2 * ref.abs() + 1.2 * (u[:, :N // 2] * u[:, N // 2:]).abs())
    else:
        ref = torch.nn.functional.gelu(u, approximate="tanh" if epi == 2 else "none")
        bound = EPS[dtype] * (ref.abs() + 1.2 * u.abs())
    _near(y, ref, 1.1 * bound + 1e-5)                        # 1e-5: the fp32 sums and functions
