"""The gated norm in front of the last of three projections, in their launch (gemv_f32.hip), against float64: widths beside a wave's
256 k, the row counts that it takes, gates that are columns of a wider row."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("sizes", [((1024, 4096), (1024, 1024), (1024, 1024)), ((5, 4), (1, 260), (130, 1020)), ((16, 64), (3, 2052), (7, 4)),
                                   ((64, 256), (64, 256), (2048, 2048))])
@pytest.mark.parametrize("small", [False, True])
def test_gated_norm_of_the_last_input(cuda, M, sizes, small):
    from edgellm import ops
    g = torch.Generator().manual_seed(M)
    xs = [torch.randn(M, K, generator=g).cuda() for _, K in sizes]
    ws = [(torch.randn(N, K, generator=g) * K ** -0.5).cuda() for N, K in sizes]
    if small:
        xs[2] *= 1e-3                                       # the norm's eps counts
    K = sizes[2][1]
    z = torch.randn(M, K + 12, generator=g).cuda()[:, 8:8 + K]
    nw = (1 + torch.rand(K, generator=g)).cuda()
    ns = [N for N, _ in sizes]
    ys = ops.ext().gemv_rows3(xs[0], ws[0], xs[1], ws[1], xs[2], ws[2], *ns, z, nw, 1e-6)
    plain = ops.ext().gemv_rows3(xs[0], ws[0], xs[1], ws[1], xs[2], ws[2], *ns)
    assert torch.equal(ys[0], plain[0]) and torch.equal(ys[1], plain[1])
    v = xs[2].double() * torch.nn.functional.silu(z.double())
    u = v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + 1e-6) * nw.double()
    ref = u @ ws[2].double().t()
    # K products of terms that carry some 8 roundings (exponential, gate, weight, the sum of squares' half) and their sum
    assert ((ys[2].double() - ref).abs() <= 2.0 ** -24 * (K + 16) * (u.abs() @ ws[2].double().abs().t()) + 1e-9).all()


def test_what_the_launch_takes(cuda):
    """Dense fp32 rows; a gate of strided columns, other layouts and types run apart."""
    from edgellm.engine.ragged_bench import hybrid_config
    from edgellm.models import mixers
    from edgellm.models.hybrid import build_hybrid
    cfg = hybrid_config(dict(width=256, layers=2, heads=4, kv=2, dim=64, window=64, pool=16, s_heads=4, s_vdim=64, state=64, ff=512, vocab=512))
    model = build_hybrid(cfg, dtype=torch.float32, device="cuda", seed=1)
    x = torch.randn(2, 256, device="cuda")
    m = model.layers[0].mix
    y, z = torch.randn(2, 256, device="cuda"), torch.randn(2, 300, device="cuda")[:, 4:260]
    assert mixers.rows_gated((x, x, y), (m.left.o, m.left.o, m.right.o), z, m.right.norm_w, 1e-6) is not None
    assert mixers.rows_gated((x, x, y), (m.left.o, m.left.o, m.right.o), z.t().contiguous().t(), m.right.norm_w, 1e-6) is None
    assert mixers.rows_gated((x, x, y.t().contiguous().t()), (m.left.o, m.left.o, m.right.o), z, m.right.norm_w, 1e-6) is None
    assert mixers.rows_gated((x, x, y), (m.left.o, m.left.o, m.right.o), z.bfloat16(), m.right.norm_w, 1e-6) is None
    x5, y5, z5 = x[:1].repeat(5, 1), y[:1].repeat(5, 1), z[:1].repeat(5, 1)              # more rows: the norm in a launch of its own
    assert mixers.rows_gated((x5, x5, y5), (m.left.o, m.left.o, m.right.o), z5, m.right.norm_w, 1e-6) is None
