"""The chunked gated linear attention (gla.hip) at the edges of its tiles against a float64 recurrence: heads beside 64 and 128 columns
and channels, scans of four numbers and of one, more chunks than the scan requests at once, portions that end inside a block, several
sequences, a state that continues, sizes and alignments that the 16-byte loads do not take."""
import pytest
import torch

import edgellm.ops.seqmix as S

pytestmark = pytest.mark.gpu


def _reference(u, a2, b, nw, state, seqs, H, N, P, tau, eps):
    u, a2, b, nw, st = (t.double().cpu() for t in (u, a2, b, nw, state))
    HN, HP = H * N, H * P
    la = torch.nn.functional.logsigmoid(u[:, 2 * HN + 2 * HP:] @ a2.T + b).view(-1, H, N) / tau
    out, at = torch.empty(u.shape[0], HP, dtype=torch.float64), 0
    for slot, start, n in seqs:
        x, s = u[at:at + n], st[slot].clone() if start else torch.zeros_like(st[slot])
        q, k, v = x[:, :HN].view(n, H, N) * N ** -0.5, x[:, HN:2 * HN].view(n, H, N), x[:, 2 * HN:2 * HN + HP].view(n, H, P)
        o = torch.empty(n, H, P, dtype=torch.float64)
        for t in range(n):
            s = la[at + t].exp()[:, :, None] * s + k[t][:, :, None] * v[t][:, None, :]
            o[t] = torch.einsum("hnp,hn->hp", s, q[t])
        o = o * torch.rsqrt(o.pow(2).mean(-1, keepdim=True) + eps) * nw
        out[at:at + n] = o.reshape(n, HP) * torch.nn.functional.silu(x[:, 2 * HN + HP:2 * HN + 2 * HP])
        st[slot], at = s, at + n
    return out, st


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,N,P,rank,seqs", [
    (2, 64, 64, 16, [(1, 0, 65)]), (1, 128, 128, 16, [(0, 0, 64), (2, 7, 130)]), (2, 72, 72, 5, [(0, 5, 79)]), (1, 8, 8, 17, [(1, 3, 1300)]),
    (1, 136, 136, 16, [(0, 9, 100)]), (3, 40, 128, 16, [(2, 0, 24), (0, 0, 1), (1, 1, 63)]), (2, 20, 30, 3, [(0, 4, 200)]),
    (1, 64, 70, 16, [(1, 2, 90), (0, 0, 33)])])
def test_chunks_at_the_edges_of_their_tiles(cuda, dt, H, N, P, rank, seqs):
    g = torch.Generator().manual_seed(H + N + P)
    T = sum(n for _, _, n in seqs)
    u = torch.randn(T, 2 * H * N + 2 * H * P + rank, generator=g).to(dt).cuda()
    a2, b = (torch.randn(H * N, rank, generator=g) * rank ** -0.5).cuda(), torch.randn(H * N, generator=g).cuda()
    nw, state = (1 + 0.1 * torch.randn(P, generator=g)).cuda(), torch.randn(3, H, N, P, generator=g).cuda()
    want, end = _reference(u, a2, b, nw, state, seqs, H, N, P, 8.0, 1e-6)
    meta = S.RaggedMeta.build(seqs, torch.zeros(3, 1, dtype=torch.int32, device="cuda"), 64, torch.device("cuda"))
    got = S.gated_linear_attention(u, a2, b, nw, state, meta, H, N, P, 8.0, 1e-6).double().cpu()
    # fp32: sums of N and of 64 terms and decays of a few roundings each, in a norm over the row; bf16: the result's rounding (2^-9 rms at most)
    tol = 2e-6 if dt == torch.float32 else 2.0 ** -9
    assert (got - want).norm() < tol * want.norm()
    assert (state.double().cpu() - end).norm() < 2e-6 * end.norm()


@pytest.mark.parametrize("N,P", [(64, 64), (20, 30)])        # scans of four numbers and of one
def test_portions_without_a_token(cuda, N, P):
    """They read no row of the chunks' states (the first one's would lie in front of them), keep a state that continues and clear one
    that starts."""
    H, rank, seqs = 2, 8, [(2, 5, 0), (0, 3, 130), (3, 0, 0), (1, 0, 70), (4, 9, 0)]
    g = torch.Generator().manual_seed(N)
    u = torch.randn(200, 2 * H * N + 2 * H * P + rank, generator=g).cuda()
    a2, b = (torch.randn(H * N, rank, generator=g) * rank ** -0.5).cuda(), torch.randn(H * N, generator=g).cuda()
    nw, state = (1 + 0.1 * torch.randn(P, generator=g)).cuda(), torch.randn(5, H, N, P, generator=g).cuda()
    want, end = _reference(u, a2, b, nw, state, seqs, H, N, P, 8.0, 1e-6)
    meta = S.RaggedMeta.build(seqs, torch.zeros(5, 1, dtype=torch.int32, device="cuda"), 64, torch.device("cuda"))
    got = S.gated_linear_attention(u, a2, b, nw, state, meta, H, N, P, 8.0, 1e-6).double().cpu()
    assert (got - want).norm() < 2e-6 * want.norm()
    assert (state.double().cpu() - end).norm() < 2e-6 * end.norm()
    assert torch.equal(state[[2, 4]].double().cpu(), end[[2, 4]]) and not state[3].any()
