"""Split-K W8A8 GEMV of up to 16 rows with a scale per (row, 64 numbers) (gemv_i8_rows.hip), against float64."""
import pytest
import torch

from edgellm import ops

pytestmark = pytest.mark.gpu


# fewer k-tiles than waves, ragged rounds and parts, one tile, many tiles, more than 16 MB whose 5 to 16 rows keep two tiles a workgroup
# (4096 x 11008) or take one (5120 x 4160)
@pytest.mark.parametrize("M", [1, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("N,K,S", [(16, 64, 0), (48, 1088, 3), (2064, 2560, 0), (4096, 11008, 2), (1024, 192, 3), (5120, 4160, 0)])
def test_slices_sum_to_the_product(cuda, M, N, K, S):
    g = torch.Generator(device=cuda).manual_seed(M * 1009 + N + K)
    ints = lambda *s: torch.randint(-127, 128, s, generator=g, device=cuda, dtype=torch.int8)  # noqa: E731
    x, w = ints(M, K), ints(N, K)
    sx = torch.rand(K // 64, 16, generator=g, device=cuda) * 0.02 + 1e-3
    sw = torch.rand(N, generator=g, device=cuda) * 1e-3 + 1e-4
    bias = torch.randn(N, generator=g, device=cuda).bfloat16()
    part = ops.ext().w8a8_gemm_splitk(x, sx, ops.pack_int8_weight(w), sw, bias, N, K, S)
    xs = x.double().view(M, K // 64, 64) * sx.double().t()[:M, :, None]
    xs = xs.reshape(M, K)
    ref = xs @ w.double().t() * sw.double() + bias.double()
    # a 64-number product is exact; its scaling and every sum round once: at most K / 64 + 16 + S + 3 steps of half an ulp of
    # what has been added up
    size = xs.abs() @ w.double().abs().t() * sw.double() + bias.double().abs()
    err = (part.double().sum(0) - ref).abs()
    assert part.shape[1:] == (M, N) and (S == 0 or part.shape[0] == S)
    assert bool((err <= (K // 64 + 24) * 2.0 ** -24 * size).all()), float((err / size).max())
