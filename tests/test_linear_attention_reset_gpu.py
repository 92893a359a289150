"""Gated linear attention whose decay is 0 for some tokens or channels (log decay -inf: a bias of the type's lowest value, a gate that
overflows), in chunks and token by token, against float64: what lies before such a token is gone, what follows it decays as it should."""
import pytest
import torch

import edgellm.ops.seqmix as S

pytestmark = pytest.mark.gpu
LOWEST = torch.finfo(torch.float32).min


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("L,H,N,P", [(7, 2, 32, 16), (70, 2, 64, 64), (200, 1, 40, 72), (131, 2, 128, 128)])
@pytest.mark.parametrize("tau", [1.0, 16.0])
def test_decays_of_zero(dt, L, H, N, P, tau):
    g = torch.Generator().manual_seed(L + N)
    HN, HP, R = H * N, H * P, 2
    u = torch.randn(L, 2 * HN + 2 * HP + R, generator=g).to(dt)
    a2, b = torch.randn(HN, R, generator=g), 2 + torch.randn(HN, generator=g)
    # the second decay input is 0 but at a few tokens (a block's first, middle and last among them), where every third channel overflows
    at = [t for t in (0, 5, 16, 31, 40, 69, 128, 130) if t < L]
    u[:, -1] = 0
    u[at, -1] = -8
    a2[:, 1] = 0
    a2[::3, 1] = -LOWEST
    b[1::7] = LOWEST                                         # channels that forget at every token
    norm_w = 1 + 0.2 * torch.randn(P, generator=g)
    state = torch.randn(2, H, N, P, generator=g)
    table = torch.zeros(2, 1, dtype=torch.int32, device="cuda")
    st = state.cuda()
    meta = S.RaggedMeta.build([(1, 3, L)], table, 512, "cuda")
    got = S.gated_linear_attention(u.cuda(), a2.cuda(), b.cuda(), norm_w.cuda(), st, meta, H, N, P, tau, 1e-5)
    x = u.double()
    z = (x[:, -R:].float() @ a2.t() + b).double()            # (overflows in fp32, as it does in the model)
    a = torch.exp(torch.nn.functional.logsigmoid(z) / tau).view(L, H, N)
    q, k, v = x[:, :HN].view(L, H, N) * N ** -0.5, x[:, HN:2 * HN].view(L, H, N), x[:, 2 * HN:2 * HN + HP].view(L, H, P)
    M, o = state[1].double(), torch.empty(L, H, P, dtype=torch.float64)
    for t in range(L):
        M = M * a[t][:, :, None] + k[t][:, :, None] * v[t][:, None, :]
        o[t] = torch.einsum("hn,hnp->hp", q[t], M)
    y = o * torch.rsqrt(o.pow(2).mean(-1, keepdim=True) + 1e-5) * norm_w.double()
    ref = y.view(L, HP) * torch.nn.functional.silu(x[:, 2 * HN + HP:2 * HN + 2 * HP])
    # fp32 sums of N + 64 products of about 1, which the norm may magnify by a few; one rounding of the result
    tol = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -14
    assert torch.isfinite(got).all()
    assert ((got.cpu().double() - ref).abs() <= tol * (1 + ref.abs())).all()
    assert ((st[1].cpu().double() - M).abs() <= 2.0 ** -17 * (1 + M.abs().max())).all()
