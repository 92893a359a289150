"""A decode step's attention and state-space recurrence in one launch (attn_step.hip's attn_ssd_kernel) against the two ops on the CPU:
both types, head sizes on both sides of a row layout, state sizes, an odd number of kv heads and rows beside the eight dies, windows with
and without blocks, gates, sequences that start and that go on, and the calls that stay two launches."""
import pytest
import torch

import edgellm.ops.seqmix as S

pytestmark = pytest.mark.gpu
PAGE = 16


def _run(dt, H, G, D, Dv, lens, window, pool, gated, Hs, P, N, groups, dev, seed=0):
    g = torch.Generator().manual_seed(seed)
    n, per = len(lens), (max(lens) + PAGE - 1) // PAGE
    rnd = lambda *s, t=dt: torch.randn(*s, generator=g).to(t)
    table = torch.randperm(n * per, generator=g).view(n, per).int()
    k, v, q = rnd(n * per, PAGE, G, D), rnd(n * per, PAGE, G, Dv), rnd(n, H, D)
    kb, vb = (rnd(n * per, PAGE // pool, G, D, t=torch.float32), rnd(n * per, PAGE // pool, G, Dv, t=torch.float32)) if pool else (None, None)
    C = Hs * P + 2 * groups * N
    xbc, u, gate = rnd(n, C), rnd(n, 24 + Hs), rnd(n, H)
    state = rnd(n + 1, Hs, N, P, t=torch.float32)
    consts = [rnd(Hs, t=torch.float32) for _ in range(3)]
    # on the CPU in fp32 over the same values
    f = dt if dev == "cuda" else torch.float32
    to = lambda t: None if t is None else t.to(dev).to(f if t.dtype == dt else t.dtype)
    st = state.to(dev)
    m = S.RaggedMeta.build([(n - i, l - 1, 1) for i, l in enumerate(lens)], torch.cat([table[:1], table.flip(0)]).to(dev), PAGE, dev)
    out = S.attention_beside_scan(to(q), to(gate) if gated else None, to(k), to(v), to(kb), to(vb), m, D ** -0.5, window, pool or None, to(xbc),
                                  to(u), 24, *[to(c) for c in consts], st, Hs, P, N, groups)
    return [t.float().cpu() for t in (*out, st)]


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,G,D,Dv,lens,window,pool,gated,Hs,P,N,groups", [
    (16, 4, 64, 64, [777, 1], 512, 16, True, 16, 64, 64, 1),
    (6, 3, 72, 40, [129, 16, 300], None, 0, False, 6, 64, 128, 2),
    (4, 1, 8, 8, [1], 5, 0, True, 2, 128, 64, 1),
    (5, 5, 128, 128, [40, 200, 17, 128, 33, 90, 1, 61, 75], 64, 4, True, 4, 128, 128, 4),
    (3, 3, 64, 64, [50], 20, 0, False, 3, 64, 64, 1),        # an odd number of state heads: two launches
    (4, 2, 64, 64, [50, 9], 20, 0, False, 2, 32, 64, 1),     # a state that the step kernel does not take: two launches
    (16, 2, 160, 64, [70], None, 0, True, 2, 64, 64, 1)])    # rows past 128 numbers: two launches
def test_side_by_side(dt, H, G, D, Dv, lens, window, pool, gated, Hs, P, N, groups):
    args = (dt, H, G, D, Dv, lens, window, pool, gated, Hs, P, N, groups)
    got, ref = _run(*args, "cuda"), _run(*args, "cpu")
    # heads: one rounding of the result, fp32 sums of weight 1 over values of about 1; y and the state: sums of up to 2 N + 1 products of
    # about 1 (rounded to 2^-24 each) that e^(A dt) scales by 1 at most
    eps = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -17
    assert ((got[0] - ref[0]).abs() <= eps * ref[0].abs() + 2.0 ** -17).all(), (got[0] - ref[0]).abs().max()
    for a, r in zip(got[1:], ref[1:]):
        assert torch.isfinite(a).all()
        assert ((a - r).abs() <= 2.0 ** -16 * r.abs().max()).all(), (a - r).abs().max()
