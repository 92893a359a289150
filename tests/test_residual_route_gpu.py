"""A residual sum with the next row's convolution and its choice of experts in one launch (residual_next.hip) against the separate
launches, bit for bit: widths at the edges of a wave's 256 columns and of its 512 of the router's, experts up to 16, every mode, and
the calls that stay apart."""
import pytest
import torch

import edgellm.ops.seqmix as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("mode", ["softmax", "sigmoid", "top_softmax"])
@pytest.mark.parametrize("T,W,E,top,bias,apart", [
    (4, 1024, 16, 3, False, False), (1, 256, 1, 1, True, False), (3, 264, 15, 15, False, False), (5, 520, 9, 2, True, False),
    (256, 512, 16, 3, False, False), (2, 1016, 12, 12, False, False),
    (2, 1032, 16, 3, False, True), (2, 1024, 17, 3, True, True), (257, 256, 16, 3, False, True), (2, 260, 16, 2, False, True)])
def test_with_the_choice(dt, mode, T, W, E, top, bias, apart):
    g = torch.Generator(device="cuda").manual_seed(W + E + T)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)
    x, y, w, b, cw, state, router = r(T, W), r(T, W).to(dt), r(W), r(W), r(W, 4), r(T + 2, 3, W), r(E, W) * W ** -0.5
    rb = r(E) if bias else None
    table = torch.zeros(T + 2, 1, dtype=torch.int32, device="cuda")
    m = S.RaggedMeta.build([(T + 1 - i, (0, 1, 2, 3, 9)[i % 5], 1) for i in range(T)], table, 16, "cuda")
    x1, x2, s1, s2 = x.clone(), x.clone(), state.clone(), state.clone()
    one = S._ext().sm_ln_residual_taps_route(x.clone(), y, w, b, 1e-5, None, None, cw, state.clone(), m.tok_seq, m.tok_pos, m.seq_slot,
                                             dt == torch.float32, router, top, 2.0, S.MOE_MODES[mode], rb)
    assert (one is None) == apart
    h1, (i1, w1) = S.layer_norm_residual_canon_route(x1, y, w, b, 1e-5, cw, s1, m, dt, router, top, 2.0, mode, rb)
    h2 = S.layer_norm_residual_canon(x2, y, w, b, 1e-5, None, None, cw, s2, m, dt)
    i2, w2 = S.moe_route(h2, router, top, 2.0, mode, rb)
    # the same sums in the same order: a product and a sum may be one rounding here and two there (2^-24 of a row's numbers of up to
    # 16; the row's type rounds them to a neighbour at most), and a choice only differs where two scores are as near as that
    eps = 2.0 ** -20
    for a, c in ((x1, x2), (s1, s2)):
        assert ((a - c).abs() <= eps * (1 + c.abs())).all()
    assert ((h1.float() - h2.float()).abs() <= (2.0 ** -7 if dt == torch.bfloat16 else eps) * (1 + h2.float().abs())).all()
    if torch.equal(h1, h2):
        assert torch.equal(i1, i2) and torch.equal(w1, w2)
    else:
        same = (i1 == i2).all(1)
        assert same.float().mean() > 0.9 and torch.allclose(w1[same], w2[same], atol=1e-2)
