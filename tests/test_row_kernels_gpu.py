"""Row kernels of the post-norm layers against the same ops in fp32 on the CPU, at the edges of their vector forms (runs of four
or eight numbers, 16 lanes per head, chunks per thread) and at widths that stay with the general kernels."""
import pytest
import torch

import edgellm.ops.seqmix as S

pytestmark = pytest.mark.gpu
DT = [torch.bfloat16, torch.float32]


def _rand(g, *s):
    return torch.randn(*s, generator=g)


def _pair(x, dt):
    """The operand on the GPU in dt and the same numbers in fp32 on the CPU."""
    return (None, None) if x is None else (x.to(dt).cuda(), x.to(dt).float())


def _near(got, ref, dt, scale=1.0):
    # fp32 sums of up to 4096 terms in another order and device exp / rsqrt (1e-6 of the row's size each), one rounding to dt
    tol = 1e-5 * scale + (2.0 ** -8 if dt == torch.bfloat16 else 1e-5) * ref.abs()
    assert ((got.float().cpu() - ref).abs() <= tol).all()


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("W", [4, 252, 256, 1020, 1024, 1028, 2048, 4096, 4100, 1022])
@pytest.mark.parametrize("T,K,with_y", [(3, 0, True), (1, 1, False), (5, 3, True), (2, 4, False), (2, 5, True), (2, 9, False)])
def test_layer_norm_residual(dt, W, T, K, with_y):
    g = torch.Generator().manual_seed(W + K)
    x, w, b = _rand(g, T, W), _rand(g, W), _rand(g, W)
    y, yc = _pair(_rand(g, T, W) if with_y else None, dt)
    parts, pc = _pair(_rand(g, T, K, W) if K else None, dt)
    pw = _rand(g, T, K) if K else None
    got = S.layer_norm_residual(x.cuda(), y, w.cuda(), b.cuda(), 1e-6, parts, pw.cuda() if K else None)
    _near(got, S.layer_norm_residual(x.clone(), yc, w, b, 1e-6, pc, pw), torch.float32, 10.0)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("heads,P,act", [(1, 4, "silu"), (16, 64, "sigmoid"), (5, 68, "silu"), (3, 128, "sigmoid"), (2, 256, "silu"),
                                         (2, 260, "sigmoid"), (3, 62, "silu")])
@pytest.mark.parametrize("T,pad", [(1, 0), (7, 4), (7, 3), (1025, 4)])
def test_head_norm_gate(dt, heads, P, act, T, pad):
    g = torch.Generator().manual_seed(P)
    y, w = _rand(g, T, heads * P), _rand(g, P)
    z, zc = _pair(_rand(g, T, heads * P + pad), dt)
    z, zc = z[:, pad:], zc[:, pad:]
    out = S.head_norm_gate(y.cuda(), z, w.cuda(), heads, 1e-6, dt, act)
    _near(out, S.head_norm_gate(y, zc, w, heads, 1e-6, torch.float32, act), dt)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("per_head", [False, True])
@pytest.mark.parametrize("heads,kv,N", [(4, 1, 4), (16, 16, 64), (8, 4, 68), (12, 6, 128), (4, 2, 256), (18, 9, 60), (3, 3, 64), (4, 2, 62),
                                        (4, 2, 260)])
def test_delta_prepare(dt, per_head, heads, kv, N):
    g = torch.Generator().manual_seed(N)
    T, C = 5, 2 * kv * N + heads * 8
    (qkv, qc), (u, uc) = _pair(_rand(g, T, C), dt), _pair(_rand(g, T, 2 * heads + 8), dt)
    bias, A = _rand(g, heads if per_head else heads * N), _rand(g, heads)
    bias[0] = 25.0
    if per_head:
        got = S.delta_prepare_head(qkv, u, 3, heads + 5, bias.cuda(), A.cuda(), heads, kv, N)
        ref = S.delta_prepare_head(qc, uc, 3, heads + 5, bias, A, heads, kv, N)
    else:
        a = _rand(g, T, heads * N)
        got = S.delta_prepare(qkv, u, 3, a.cuda(), bias.cuda(), A.cuda(), heads, kv, N)
        ref = S.delta_prepare(qc, uc, 3, a, bias, A, heads, kv, N)
    _near(got, ref, torch.float32)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("H,D,R,kvr,rot", [(16, 64, 32, 128, 32), (3, 8, 8, 8, 0), (33, 8, 8, 8, 0), (5, 16, 16, 24, 8), (13, 16, 16, 24, 8), (2, 128, 64, 256, 64), (3, 12, 8, 16, 8), (33, 12, 8, 16, 8),
                                           (2, 8, 6, 10, 4), (2, 8, 8, 16, 4)])
def test_latent_write(dt, H, D, R, kvr, rot):
    g = torch.Generator().manual_seed(H)
    seqs = [(1, 60, 7), (0, 0, 3)]
    tab = torch.tensor([[2, 0], [1, 3]], dtype=torch.int32)
    u, q, ql, w = _rand(g, 10, kvr + R + 3), _rand(g, 10, H, D + R), _rand(g, H, 10, kvr), _rand(g, kvr)
    ang = _rand(g, 80, max(rot // 2, 1))
    rope = torch.stack([ang.cos(), ang.sin()], -1).contiguous()
    res = []
    for dev, t in (("cuda", dt), ("cpu", torch.float32)):
        meta = S.RaggedMeta.build(seqs, tab.to(dev), 64, torch.device(dev))
        pages = torch.zeros(4, 64, 1, kvr + R, dtype=t, device=dev)
        cast = lambda x: x.to(dt).to(dev, t)
        qc = S.latent_write(cast(u), 3, w.to(dev), 1e-6, cast(q), cast(ql).transpose(0, 1), meta, rope.to(dev) if rot else None,
                            pages, kvr, rot)
        res.append((qc.reshape(10, -1), pages))
    _near(res[0][0], res[1][0].cpu(), dt)
    _near(res[0][1], res[1][1].cpu(), dt)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("H,D,R,kvr,rot", [(16, 64, 32, 128, 32), (3, 8, 8, 8, 0), (2, 128, 64, 256, 64), (2, 8, 6, 10, 4), (1, 1, 2, 1, 2)])
@pytest.mark.parametrize("T", [1, 16, 17])
def test_queries_of_shared_latents(dt, H, D, R, kvr, rot, T):
    """Queries against another layer's cached rows: up to 16 tokens in one launch, 17 in two; the rows stay as they are."""
    g = torch.Generator().manual_seed(H + T)
    tab = torch.arange(T, dtype=torch.int32).view(T, 1)
    q, uk = _rand(g, T, H, D + R), _rand(g, H, D, kvr) * D ** -0.5
    ang = _rand(g, 80, max(rot // 2, 1))
    rope, rows = torch.stack([ang.cos(), ang.sin()], -1).contiguous(), _rand(g, T, 64, 1, kvr + R)
    res = []
    for dev, t in (("cuda", dt), ("cpu", torch.float32)):
        meta = S.RaggedMeta.build([(i, i, 1) for i in range(T)], tab.to(dev), 64, torch.device(dev))
        cast = lambda x: x.to(dt).to(dev, t)
        pages = cast(rows)
        qc = S.latent_expand_write(None, 0, None, 1e-6, cast(q), cast(uk), meta, rope.to(dev) if rot else None, pages, kvr, rot)
        assert torch.equal(pages, cast(rows))
        res.append(qc.reshape(T, -1))
    _near(res[0], res[1].cpu(), dt)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("T,E,W,bias", [(64, 16, 1024, False), (768, 16, 1024, False), (2459, 5, 520, True), (374, 33, 2048, False),
                                        (12289, 1, 8, True), (770, 16, 1030, False)])
def test_router_scores_of_prompts(dt, T, E, W, bias):
    """From 12288 scores on four tokens share the router's rows: the same choices and weights, bit for bit, as in small steps."""
    g = torch.Generator().manual_seed(E)
    h, router = _rand(g, T, W).to(dt).cuda(), _rand(g, E, W).cuda()
    b = _rand(g, E).cuda() if bias else None
    top = min(3, E)
    idx, wts = S.moe_route(h, router, top, 1.5, "softmax", b)
    small = [S.moe_route(h[a:a + 63].contiguous(), router, top, 1.5, "softmax", b) for a in range(0, T, 63)]
    assert torch.equal(idx, torch.cat([s[0] for s in small])) and torch.equal(wts, torch.cat([s[1] for s in small]))
