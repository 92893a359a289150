"""One-row int8 projections at the edges of their tiles per workgroup (gemm_i8.hip launch_norm_out: 1, 2 or 3 column
tiles by N), and the row that LLM.int8 adds in the epilogue: each against the unfused form, bit for bit."""
import pytest
import torch

import edgellm.ops as ops

pytestmark = pytest.mark.gpu

EDGES = [16, 16 * 255, 16 * 256, 16 * 257, 16 * 512, 16 * 513, 16 * 515]


@pytest.fixture
def cuda():
    return torch.device("cuda:0")


def _l8(N, K, dev):
    from edgellm.models.layers import Linear
    from edgellm.quant import LLMInt8Linear
    lin = Linear(K, N, bias=True, device=dev)
    lin.weight.data.copy_(torch.randn(N, K, device=dev) * 0.02)
    lin.bias.data.copy_(torch.randn(N, device=dev) * 0.1)
    return LLMInt8Linear.from_float(lin)


@pytest.mark.parametrize("N", EDGES)
@pytest.mark.parametrize("K,where", [(64, []), (2112, [0, 63, 2047, 2048, 2111]), (4096, range(0, 4096, 3)),
                                     (12288, [5, 2049, 6000, 8191, 8192, 12287])])
def test_llmint8_tiles_and_added_row(cuda, N, K, where):
    """The one-launch LLM.int8 row (+ the added row) == the three-launch path, then the sum: outliers in every chunk of
    2048 columns, past the 256-column cap, and none."""
    torch.manual_seed(N + K)
    m = _l8(N, K, cuda)
    x = torch.randn(1, K, device=cuda)
    x[0, list(where)] = 9.0
    x = x.bfloat16()
    add = torch.randn(1, 1, N, device=cuda).bfloat16()
    one, summed = m(x), m(x.view(1, 1, K), add=add)
    wide = torch.randn(1, 2 * N, device=cuda).bfloat16()[:, ::2]            # not dense: added outside the launch
    strided = m(x, add=wide)
    m.ONE_LAUNCH = False
    ref = m(x)
    assert torch.equal(one, ref)
    assert torch.equal(summed, ref.view_as(summed) + add) and torch.equal(strided, ref + wide)


@pytest.mark.parametrize("rows", [3, 70])
def test_llmint8_added_rows(cuda, rows):
    """More rows than the one-launch form takes: the sum is kept."""
    torch.manual_seed(rows)
    m = _l8(96, 128, cuda)
    x, add = torch.randn(rows, 128, device=cuda).bfloat16(), torch.randn(rows, 96, device=cuda).bfloat16()
    assert torch.equal(m(x, add=add), m(x) + add)


@pytest.mark.parametrize("N", EDGES)
@pytest.mark.parametrize("kind,K", [("rms", 2048), ("rms", 4096), ("ln", 2048), ("ln", 2560)])
def test_w8a8_norm_prologue_tiles(cuda, N, kind, K):
    """W8A8 rows normed in the prologue == the norm kernel, then the projection."""
    torch.manual_seed(N + K)
    w = torch.randint(-127, 128, (N, K), dtype=torch.int8, device=cuda)
    wp = ops.pack_int8_weight(w)
    sw = torch.rand(N, device=cuda) * 0.004 + 1e-4
    bias = torch.randn(N, device=cuda).bfloat16()
    gamma = (torch.rand(K, device=cuda) + 0.5).bfloat16()
    for M in (1, 2):
        res = torch.randn(M, K, device=cuda).bfloat16()
        h = torch.empty_like(res)
        if kind == "rms":
            parts = torch.randn(2, M, K, device=cuda)
            q, s, _ = ops.rms_norm_parts(parts, res, gamma, 1e-5, True)
            out = ops.w8a8_gemv_norm(parts, res, gamma, 1e-5, h, wp, sw, bias, N, K)
        else:
            beta, x = torch.randn(K, device=cuda).bfloat16(), torch.randn(M, K, device=cuda).bfloat16()
            q, s, _ = ops.layer_norm_quant(x, gamma, beta, 1e-5, res)
            out = ops.w8a8_gemv_ln(x, res, gamma, beta, 1e-5, h, wp, sw, bias, N, K)
        assert out is not None and torch.equal(out, ops.w8a8_linear(q, s, wp, sw, bias, N, K))
