"""A gated delta rule's decode step in one launch (delta_step.hip) against the separate ops in fp32 on the CPU: both kinds of
decays, both head sizes, steps from positions 0 to 3 and later, several steps in a row (tail and state move on), and the calls
that stay with the separate kernels."""
import pytest
import torch

import edgellm.ops.seqmix as S

pytestmark = pytest.mark.gpu


def _apart(u, b0, a0, z0, a2, g2, conv_w, conv_b, tail, state, dt_bias, A_log, norm_w, eps, meta, H):
    N, P = state.shape[2:]
    C = conv_w.shape[0]
    qkv = S.conv_silu(u, 0, C, conv_w, conv_b, tail, meta)
    if a2 is None:
        prep, z, act = S.delta_prepare_head(qkv, u, b0, a0, dt_bias, A_log, H, H, N), u[:, z0:z0 + H * P], "silu"
    else:
        a = u[:, a0:a0 + a2.shape[1]].float() @ a2.float().t()
        z, act = (u[:, z0:z0 + g2.shape[1]].float() @ g2.float().t()).to(u.dtype), "sigmoid"
        prep = S.delta_prepare(qkv, u, b0, a, dt_bias, A_log, H, H, N)
    y = S.delta_rule_scan(prep, qkv, state, meta, H, H, N, P)
    return S.head_norm_gate(y, z, norm_w, H, eps, u.dtype, act)


def _case(dt, H, N, P, ra, rg, n, seed):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g)
    C = 2 * H * N + H * P
    width = C + H + (ra + rg if ra else H + H * P)
    u = [r(n, width).to(dt) for _ in range(3)]
    w = dict(a2=r(H * N, ra).to(dt) * ra ** -0.5 if ra else None, g2=r(H * P, rg).to(dt) * rg ** -0.5 if rg else None, conv_w=r(C, 4) * 0.5,
             conv_b=r(C) * 0.1, dt_bias=r(H * N if ra else H), A_log=r(H) * 0.5, norm_w=r(P))
    return u, w, r(n + 2, 3, C).to(dt), r(n + 2, H, N, P), C, torch.randperm(n + 2, generator=g)[:n].tolist()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,N,P,ra,rg", [(16, 64, 64, 32, 32), (3, 64, 64, 0, 0), (8, 64, 64, 0, 0), (16, 128, 128, 64, 64), (2, 128, 128, 0, 0),
                                         (8, 128, 128, 8, 136)])
@pytest.mark.parametrize("n", [1, 5])
def test_steps(dt, H, N, P, ra, rg, n):
    us, w, tail, state, C, slots = _case(dt, H, N, P, ra, rg, n, H + N + ra)
    starts = [(0, 1, 2, 3, 40)[i % 5] for i in range(n)]
    for s, p in zip(slots, starts):
        if p:
            tail[s, :max(0, 3 - p)] = 0                     # a tail has nothing before position 0
    tail_d, state_d, tail_c, state_c = tail.cuda(), state.cuda(), tail.clone(), state.clone()
    cols = (C, C + H, C + H + (ra or H))
    table = torch.zeros(n + 2, 1, dtype=torch.int32)
    for i, u in enumerate(us):
        seqs = [(s, p + i, 1) for s, p in zip(slots, starts)]
        cu = lambda t: None if t is None else t.cuda()
        wide = torch.zeros(n, u.shape[1] + 8, dtype=dt, device="cuda")            # rows that lie apart
        wide[:, :u.shape[1]] = u.cuda()
        got = S.delta_step(wide[:, :u.shape[1]], *cols, cu(w["a2"]), cu(w["g2"]), cu(w["conv_w"]), cu(w["conv_b"]), tail_d, state_d,
                           cu(w["dt_bias"]), cu(w["A_log"]), cu(w["norm_w"]), 1e-6, S.RaggedMeta.build(seqs, table.cuda(), 16, "cuda"), H)
        ref = _apart(u, *cols, w["a2"], w["g2"], w["conv_w"], w["conv_b"], tail_c, state_c, w["dt_bias"], w["A_log"], w["norm_w"], 1e-6,
                     S.RaggedMeta.build(seqs, table, 16, "cpu"), H)
        # fp32 sums of up to 136 and 128 terms in another order; bf16: silu's rounding may fall to the neighbour in q | k | v
        eps = 2.0 ** -6 if dt == torch.bfloat16 else 1e-4
        assert (got.float().cpu() - ref.float()).abs().max() <= eps * ref.float().abs().max()
        assert torch.equal(tail_d.cpu(), tail_c)
        assert (state_d.cpu() - state_c).abs().max() <= eps * state_c.abs().max()


def test_what_stays_apart():
    us, w, tail, state, C, slots = _case(torch.bfloat16, 4, 64, 64, 0, 0, 2, 1)
    d = lambda t: None if t is None else t.cuda()
    table = torch.zeros(4, 4, dtype=torch.int32, device="cuda")
    args = lambda u, st, m, kv: S.delta_step(u, C, C + 4, C + 8, None, None, d(w["conv_w"]), d(w["conv_b"]), d(tail), st, d(w["dt_bias"]),
                                             d(w["A_log"]), d(w["norm_w"]), 1e-6, m, kv)
    one = S.RaggedMeta.build([(0, 5, 1), (1, 3, 1)], table, 16, "cuda")
    two = S.RaggedMeta.build([(0, 5, 2)], table, 16, "cuda")
    assert args(us[0].cuda(), d(state), one, 4) is not None
    assert args(us[0].cuda(), d(state), one, 2) is None                       # shared q and k
    assert args(us[0].cuda(), d(state), two, 4) is None                       # a portion of two tokens


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,pad", [(3, 8), (8, 4)])          # the decay's rows start off eight numbers; rows lie off eight numbers apart
def test_low_rank_rows_off_16_bytes_stay_apart(dt, H, pad):
    us, w, tail, state, C, slots = _case(dt, H, 64, 64, 32, 32, 2, 7)
    u = us[0]
    wide = torch.zeros(2, (u.shape[1] + 7) // 8 * 8 + pad, dtype=dt, device="cuda")
    wide[:, :u.shape[1]] = u.cuda()
    d = {k: v.cuda() for k, v in w.items()}
    tail_d, state_d = tail.cuda(), state.cuda()
    m = S.RaggedMeta.build([(s, 5, 1) for s in slots], torch.zeros(4, 1, dtype=torch.int32, device="cuda"), 16, "cuda")
    assert (C + H) % 8 != 0 or wide.stride(0) % 8 != 0
    assert S.delta_step(wide[:, :u.shape[1]], C, C + H, C + H + 32, d["a2"], d["g2"], d["conv_w"], d["conv_b"], tail_d, state_d, d["dt_bias"],
                        d["A_log"], d["norm_w"], 1e-6, m, H) is None
    assert torch.equal(tail_d.cpu(), tail) and torch.equal(state_d.cpu(), state)             # nothing was done
