"""A parallel layer's parts between its input projection and its mixers in one launch (parallel_step.hip) against the separate ops
on the CPU: positions on both sides of a block's end and of the convolution's start, rows and widths beside a workgroup's 2048
numbers, no rotation, no blocks, no feed-forward, blocks that do not divide a page, and the calls that stay with the separate ops."""
import pytest
import torch

import edgellm.ops.seqmix as S

pytestmark = pytest.mark.gpu
PAGE = 16


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,G,D,Dv,rot,pool,C,F", [(16, 4, 64, 64, 64, 16, 1152, 4096), (4, 2, 40, 24, 16, 4, 8, 0), (3, 3, 16, 16, 0, 5, 2056, 2056),
                                                   (8, 1, 128, 64, 32, 0, 264, 72), (2, 1, 8, 8, 0, 1, 16, 8)])
def test_parts(dt, H, G, D, Dv, rot, pool, C, F):
    g = torch.Generator().manual_seed(H + C)
    pos = [0, 1, 2, 3, 15, 16, 31, 47, 4]
    n, per = len(pos), 4
    gate = 16                                                # columns that no part reads
    c0 = H * D + G * (D + Dv) + gate
    f0 = c0 + C + 8
    u = torch.randn(n, f0 + F, generator=g).to(dt)
    rope = torch.randn(64, rot // 2, 2, generator=g) if rot else None
    table = torch.randperm(n * per, generator=g).view(n, per).int()
    pb = (PAGE + pool - 1) // pool if pool else 0
    mk = lambda *s, t=dt: torch.randn(*s, generator=g).to(t)
    k, v = mk(n * per, PAGE, G, D), mk(n * per, PAGE, G, Dv)
    kb, vb = (mk(n * per, pb, G, D, t=torch.float32), mk(n * per, pb, G, Dv, t=torch.float32)) if pool else (None, None)
    w, b, tail = mk(C, 4, t=torch.float32), mk(C, t=torch.float32), mk(n, 3, C)
    slots = torch.randperm(n, generator=g).tolist()
    for s, p in zip(slots, pos):
        if p:
            tail[s, :max(0, 3 - p)] = 0                     # a tail has nothing before position 0
    seqs = [(s, p, 1) for s, p in zip(slots, pos)]
    to = lambda dev: [None if t is None else t.to(dev, copy=True) for t in (u, rope, k, v, kb, vb, w, b, tail)]
    du, drope, dk, dv, dkb, dvb, dw, db, dtail = to("cuda")
    m = S.RaggedMeta.build(seqs, table.cuda(), PAGE, "cuda")
    got = S.parallel_step_in(du, m, drope, dk, dv, dkb, dvb, H, rot, pool, c0, dw, db, dtail, f0, F)
    cu, crope, ck, cv, ckb, cvb, cw, cb, ctail = to("cpu")
    m = S.RaggedMeta.build(seqs, table, PAGE, "cpu")
    q = S.rope_paged_write(cu[:, :H * D + G * (D + Dv)], m, crope, ck, cv, H, rot)
    if pool:
        S.pool_blocks(ck, cv, ckb, cvb, m, pool)
    xbc = S.conv_silu(cu, c0, C, cw, cb, ctail, m)
    act = S.relu2(cu, f0, F)
    # single products and sums of up to 16 terms in fp32, one rounding to dt (bf16: it may fall to the neighbour)
    eps = 2.0 ** -7 if dt == torch.bfloat16 else 1e-5
    for a, r in zip((*got, dk, dv, dtail), (q, xbc, act, ck, cv, ctail)):
        assert a.shape == r.shape
        assert ((a.float().cpu() - r.float()).abs() <= eps * r.float().abs() + 1e-5).all()
    if pool:
        for a, r in ((dkb, ckb), (dvb, cvb)):
            assert ((a.cpu() - r).abs() <= (2.0 ** -8 if dt == torch.bfloat16 else 1e-5) * 4).all()


def test_what_stays_apart():
    u = torch.randn(2, 64 + 32 + 8, device="cuda")
    k = torch.zeros(2, PAGE, 1, 16, device="cuda")
    table = torch.zeros(2, 1, dtype=torch.int32, device="cuda")
    call = lambda uu, m, taps=4: S.parallel_step_in(uu, m, None, k, k.clone(), None, None, 2, 0, 0, 64, torch.zeros(32, taps, device="cuda"),
                                                    torch.zeros(32, device="cuda"), torch.zeros(2, taps - 1, 32, device="cuda"), 96, 8)
    one = S.RaggedMeta.build([(0, 0, 1), (1, 3, 1)], table, PAGE, "cuda")
    assert call(u, one) is not None
    assert call(u, one, 3) is None                                            # three taps
    assert call(u, S.RaggedMeta.build([(0, 0, 2)], table, PAGE, "cuda")) is None
    assert call(torch.randn(2, 105, device="cuda")[:, 1:], one) is None       # rows that do not lie on 16 bytes


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,P,N,groups", [(4, 64, 64, 1), (6, 64, 128, 3), (2, 128, 64, 2), (3, 128, 128, 1), (2, 32, 64, 1), (4, 64, 60, 2)])
def test_recurrence_of_one_token(dt, H, P, N, groups):
    """ssd_step.hip's state sizes and others, three steps in a row, positions 0 and later, step sizes on both sides of 20."""
    g = torch.Generator().manual_seed(H + P + N)
    n, inner = 5, H * P
    r = lambda *s: torch.randn(*s, generator=g)
    bias, A_log, D = r(H), r(H) * 0.3, r(H)
    bias[0] = 21.0
    state = r(n + 1, H, N, P)
    dev_state, ref_state = state.cuda(), state.clone()
    table = torch.zeros(n + 1, 1, dtype=torch.int32)
    slots = torch.randperm(n + 1, generator=g)[:n].tolist()
    for i in range(3):
        xbc, u = r(n, inner + 2 * groups * N).to(dt), r(n, H + 3).to(dt)
        seqs = [(s, j * 3 + i, 1) for j, s in enumerate(slots)]
        got = S.ssd_scan(xbc.cuda(), u.cuda(), 3, bias.cuda(), A_log.cuda(), D.cuda(), dev_state, S.RaggedMeta.build(seqs, table.cuda(), PAGE, "cuda"), H, P, N, groups)
        ref = S.ssd_scan(xbc, u, 3, bias, A_log, D, ref_state, S.RaggedMeta.build(seqs, table, PAGE, "cpu"), H, P, N, groups)
        # fp32 on both sides: sums of N products in another order, device exponentials
        assert (got.cpu() - ref).abs().max() <= 2e-5 * ref.abs().max()
        assert (dev_state.cpu() - ref_state).abs().max() <= 2e-5 * ref_state.abs().max()
