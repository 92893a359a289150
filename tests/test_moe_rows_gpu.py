"""Experts of decode-sized steps (moe_rows.h) against the same op in fp32 on the CPU: every count of tokens per expert that
the shared readings distinguish (1, 2, 3, 4, 5 and all), widths beside a wave's 512 and 1024 numbers and a workgroup's rows,
experts on both sides of the size from which readings are shared, repeated and out-of-range choices, more pairs than one
ballot names (by tokens and by choices), the shared expert, widths of the general kernels."""
import pytest
import torch

import edgellm.ops.seqmix as S

pytestmark = pytest.mark.gpu

CHOICES = {
    "one": [[2, 0]],
    "apart": [[0, 1], [2, 3], [4, 5]],
    "pairs": [[0, 1], [1, 2], [2, 0]],
    "three": [[3, 0], [3, 1], [0, 3]],
    "five": [[1, 0], [1, 2], [3, 1], [1, 4], [5, 1]],
    "all": [[4, 4], [4, 4], [4, 4], [4, 4], [4, -7], [99, 4]],
    "many": [[i % 6, (i * 5 + 1) % 6] for i in range(40)],
    "wide": [[(i + k) % 6 for k in range(8)] for i in range(9)],
}


def _operands(dt, W, ff, top, T, act, seed):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: (torch.randn(*s, generator=g) * 0.3).to(dt)
    return r(T, W), r(6, ff if act == "relu2" else 2 * ff, W), r(6, W, ff), torch.rand(T, top, generator=g) + 0.5, r(ff + 8, W), r(W, ff + 8)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("name", list(CHOICES))
@pytest.mark.parametrize("W,ff,act", [(8, 8, "glu_clamp"), (520, 24, "silu_glu"), (1024, 520, "silu_w"), (1032, 16, "glu_clamp"),
                                      (2056, 40, "silu_glu"), (512, 1032, "relu2"), (1024, 20, "silu_glu"), (20, 64, "relu2"),
                                      (1032, 1032, "silu_glu"), (1032, 1048, "relu2")])
def test_decode_sized_experts(dt, name, W, ff, act):
    """No case has both widths whole 64s: none is the grouped kernels', of whatever length."""
    T, top = len(CHOICES[name]), len(CHOICES[name][0])
    h, w_gu, w_down, in_w, su, sd = _operands(dt, W, ff, top, T, act, T + W)
    idx = torch.tensor(CHOICES[name], dtype=torch.int32)
    op, in_w = ("silu_glu", in_w) if act == "silu_w" else (act, None)
    cuda = lambda x: None if x is None else x.cuda()
    assert not S.moe_grouped(h.cuda(), idx.cuda(), w_gu.cuda(), w_down.cuda(), op, cuda(in_w))
    got = S.moe_experts(h.cuda(), idx.cuda(), w_gu.cuda(), w_down.cuda(), 1.5, op, cuda(in_w)).float().cpu()
    f = lambda x: x.float()
    ref = S.moe_experts(f(h), idx.clamp(0, 5), f(w_gu), f(w_down), 1.5, op, in_w)
    # the inner row is rounded to dt before the second product: ff terms of at most 2^-8 (2^-24) of their size each
    u = torch.stack([torch.stack([f(w_down)[e].abs() @ torch.ones(ff) for e in row.clamp(0, 5)]) for row in idx])
    inner = S.moe_experts(f(h), idx.clamp(0, 5), f(w_gu), torch.eye(ff).repeat(6, 1, 1), 1.5, op, in_w).abs().amax(-1, keepdim=True)
    eps = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -20
    assert ((got - ref).abs() <= eps * (ref.abs() + u * inner) + 1e-6).all()
    if act == "relu2":
        o, o_sh = S.moe_experts_shared(h.cuda(), idx.cuda(), w_gu.cuda(), w_down.cuda(), su.cuda(), sd.cuda())
        y = S.relu2(f(h) @ f(su).t())
        sh = y @ f(sd).t()
        assert torch.equal(o.float().cpu(), got)
        assert ((o_sh.float().cpu() - sh).abs() <= eps * (sh.abs() + f(sd).abs().sum(1) * y.amax(-1, keepdim=True)) + 1e-6).all()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("W,ff,sff", [(8, 8, 16), (1032, 24, 1048), (512, 1032, 8), (64, 512, 72)])
@pytest.mark.parametrize("T", [1, 3, 4, 5, 8, 12])
def test_clamped_shared_expert(dt, T, W, ff, sff):
    """The shared expert beside the routed ones: the routed results keep their bits, its own are those of a float64 product."""
    g = torch.Generator().manual_seed(T + W + sff)
    r = lambda *s: (torch.randn(*s, generator=g) * 0.3).to(dt)
    h, w_gu, w_down, su, sd = r(T, W), r(6, 2 * ff, W), r(6, W, ff), r(2 * sff, W), r(W, sff)
    idx = torch.randint(0, 6, (T, 2), generator=g, dtype=torch.int32)
    D = lambda x: x.cuda()
    both = S.moe_experts_glu_shared(D(h), D(idx), D(w_gu), D(w_down), 1.5, D(su), D(sd), 0.8)
    if dt == torch.float32 and T > 1:
        assert both is None
        return
    assert torch.equal(both[0], S.moe_experts(D(h), D(idx), D(w_gu), D(w_down), 1.5))
    y = S.glu_clamp(h.double() @ su.double().t(), sff, 0.8)
    ref = y @ sd.double().t()
    eps = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -20    # one rounding of the inner row and one of the result
    bound = eps * (ref.abs() + sd.double().abs().sum(1) * y.abs().amax(-1, keepdim=True)) + 1e-6
    assert ((both[1].cpu().double() - ref).abs() <= bound).all()
    assert S.moe_experts_glu_shared(D(h.repeat(13, 1)), D(idx.repeat(13, 1)), D(w_gu), D(w_down), 1.5, D(su), D(sd), 0.8) is None
