"""A residual sum with the next row's convolution and its choice of experts in one launch (residual_next.hip): the rows against the
separate launches, to a rounding, the choice and its weights against float64 scores of the very rows it wrote: widths at the edges of
a wave's 256 columns and of its 512 of the router's, experts up to 16, every mode, and the calls that stay apart."""
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
    # the same sums in the same order: a product and a sum may be one rounding here and two there (2^-24 of a row's numbers of up to
    # 16; the row's type rounds them to a neighbour at most)
    eps = 2.0 ** -20
    for a, c in ((x1, x2), (s1, s2)):
        assert ((a - c).abs() <= eps * (1 + c.abs())).all()
    assert ((h1.float() - h2.float()).abs() <= (2.0 ** -7 if dt == torch.bfloat16 else eps) * (1 + h2.float().abs())).all()
    # scores: W products and a bias added up in fp32 in any order; a softmax in front of the choice rounds a few times more (2^-20)
    z = h1.double() @ router.double().t() + (rb.double() if bias else 0.)
    d = (W + 8) * 2.0 ** -24 * (h1.double().abs() @ router.double().abs().t() + (rb.double().abs() if bias else 0.)).max(1).values + 2.0 ** -20
    assert ((i1 >= 0) & (i1 < E)).all() and (i1.sort(1).values.diff(dim=1) > 0).all()
    zc, rest = z.gather(1, i1.long()), z.scatter(1, i1.long(), -float("inf")).max(1).values
    assert (zc.diff(dim=1) <= 2 * d[:, None]).all() and (zc[:, -1] >= rest - 2 * d).all()       # largest first, none larger left out
    ref = 2. * (torch.sigmoid(zc) if mode == "sigmoid" else torch.softmax(zc, 1))
    # a score off by d moves a sigmoid by d of itself at most and a softmax by 2 d; the functions' own roundings 2^-20
    assert ((w1.double() - ref).abs() <= ref * (2.1 * d[:, None] + 2.0 ** -20)).all()
