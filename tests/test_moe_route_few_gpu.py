"""The one-launch routers of few tokens (postnorm.hip, route_few_kernel) against the rule in float64 on the CPU: expert counts
beside a wave's 16 scores each, widths beside 512 numbers a pass, ties, scores that are no numbers, both sides of the line."""
import pytest
import torch

import edgellm.ops.seqmix as S

pytestmark = pytest.mark.gpu


def _operands(dt, T, W, n, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(T, W, generator=g).to(dt), torch.randn(n, W, generator=g) * W ** -0.5, torch.randn(n, generator=g) * 0.2


def _same(got, ref, z):
    """ids as the rule says wherever the scores lie apart by more than fp32 sums may differ; weights to fp32."""
    idx, w = got[0].cpu(), got[1].cpu()
    srt = z.sort(-1, descending=True)[0]
    apart = (srt[:, :-1] - srt[:, 1:]).amin(-1) > 1e-4
    assert apart.float().mean() > 0.5
    assert torch.equal(idx[apart], ref[0][apart].int())
    assert (w.double() - ref[1].double())[apart].abs().max() <= 2e-5


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,W,E,top", [(1, 8, 1, 1), (4, 64, 4, 2), (3, 520, 16, 3), (5, 1024, 17, 4), (9, 2048, 32, 4), (2, 2040, 33, 33),
                                       (512, 256, 8, 2), (513, 256, 8, 2), (256, 2048, 47, 4), (257, 2048, 47, 4),
                                       (6, 512, 48, 8), (6, 512, 49, 8), (3, 2056, 16, 2)])
@pytest.mark.parametrize("mode", ["softmax", "sigmoid", "top_softmax"])
def test_plain(dt, T, W, E, top, mode):
    h, r, b = _operands(dt, T, W, E, T + W + E)
    z = h.double() @ r.double().t() + b.double()
    zt, idx = torch.topk(z, top, -1)
    w = torch.softmax(zt, -1) if mode == "top_softmax" else torch.sigmoid(zt) if mode == "sigmoid" else \
        torch.softmax(z, -1).gather(1, idx) / torch.softmax(z, -1).gather(1, idx).sum(-1, keepdim=True)
    _same(S.moe_route(h.cuda(), r.cuda(), top, 1.5, mode, b.cuda()), (idx, w * 1.5), z if E > 1 else torch.tensor([[1.0, 0.0]]).repeat(T, 1))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,W,E,top,groups,keep", [(1, 64, 8, 2, 4, 1), (4, 1024, 16, 3, 4, 2), (7, 2048, 32, 3, 4, 2), (3, 256, 47, 5, 1, 1),
                                                   (5, 128, 48, 4, 8, 3), (512, 64, 6, 2, 3, 2)])
@pytest.mark.parametrize("gate", [False, True])
def test_grouped(dt, T, W, E, top, groups, keep, gate):
    h, r, b = _operands(dt, T, W, E + gate, T + W + E)
    corr = b[:E]
    got = S.moe_route_grouped(h.cuda(), r.cuda(), top, 2.0, corr.cuda(), groups, keep, gate)
    ref = S.moe_route_grouped(h, r, top, 2.0, corr, groups, keep, gate)
    c = torch.softmax(h.double() @ r[:E].double().t(), -1) + corr.double()
    _same(got, ref, c)
    if gate:
        assert (got[2].cpu() - ref[2]).abs().max() <= 2e-5


def test_ties_and_no_numbers():
    h = torch.ones(3, 64, device="cuda")
    r = torch.zeros(20, 64, device="cuda")
    assert S.moe_route(h, r, 4, 1.0)[0].tolist() == [[0, 1, 2, 3]] * 3                  # the lower id on a tie
    assert S.moe_route_grouped(h, r, 4, 1.0, None, 5, 2)[0].tolist() == [[0, 1, 2, 3]] * 3
    bad = torch.full_like(r, float("nan"))
    assert S.moe_route(h, bad, 4, 1.0)[0].tolist() == [[0, 1, 2, 3]] * 3               # ids stay in range
    assert S.moe_route_grouped(h, bad, 4, 1.0, None, 5, 2)[0].tolist() == [[0, 1, 2, 3]] * 3
