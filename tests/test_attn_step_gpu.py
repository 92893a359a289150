"""Attention of steps of few queries (attn_step.hip) against the same op on the CPU, in fp32 over the operands' exact values:
head sizes beside the four row layouts, one head a workgroup and four, keys beside a wave's 16, a round's 128 and a split,
windows, kept first tokens, pooled blocks, chunks, caps, slopes, sinks, distance biases, gates and result views, and calls
that stay with the general kernel."""
import pytest
import torch

import edgellm.ops.seqmix as S

pytestmark = pytest.mark.gpu
PAGE = 16


def _meta(lens, dev, table):
    return S.RaggedMeta.build([(i, n - 1, 1) for i, n in enumerate(lens)], table.to(dev), PAGE, dev)


def _check(dt, lens, H, G, D, Dv, run, pool=0, latent=False, seed=0):
    g = torch.Generator().manual_seed(seed)
    per = (max(lens) + PAGE - 1) // PAGE
    pages = per * len(lens)
    table = torch.randperm(pages, generator=g).view(len(lens), per).int()
    k = torch.randn(pages, PAGE, G, D, generator=g).to(dt)
    v = k[..., :Dv] if latent else torch.randn(pages, PAGE, G, Dv, generator=g).to(dt)
    q = torch.randn(len(lens), H, D, generator=g).to(dt)
    kb = torch.randn(pages, PAGE // pool, G, D, generator=g) if pool else None
    vb = torch.randn(pages, PAGE // pool, G, Dv, generator=g) if pool else None

    def on(dev, f):
        c = lambda t: None if t is None else t.to(dev).to(f if t.dtype == dt else t.dtype)
        kd = c(k)
        return run(c(q), kd, kd[..., :Dv] if latent else c(v), c(kb), c(vb), _meta(lens, dev, table), c)
    got, ref = on("cuda", dt).float().cpu(), on("cpu", torch.float32)
    # one rounding of the result; fp32 sums under weights of sum 1 over values of about 1, on both sides (a key left out or taken twice
    # among some hundred changes 1 / 300 and more)
    eps = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -17
    assert torch.isfinite(got).all()
    assert ((got - ref).abs() <= eps * ref.abs() + 2.0 ** -17).all(), (got - ref).abs().max()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,G,D,Dv", [(4, 4, 8, 8), (16, 4, 64, 64), (15, 5, 80, 80), (6, 1, 72, 40), (16, 1, 160, 128), (16, 1, 320, 256),
                                      (7, 1, 200, 136), (5, 5, 128, 128), (3, 1, 20, 12), (4, 1, 328, 64)])
@pytest.mark.parametrize("lens", [[1], [16, 17, 15], [127, 128, 129, 300], [40] * 50])
def test_plain(dt, H, G, D, Dv, lens):
    gate = torch.randn(len(lens), H, generator=torch.Generator().manual_seed(1)).to(dt)
    sink = torch.linspace(-1, 3, H)
    _check(dt, lens, H, G, D, Dv, lambda q, k, v, kb, vb, m, on: S.window_pool_attention(
        q, on(gate), k, v, None, None, m, D ** -0.5, None, None, on(sink)), latent=G == 1 and Dv <= D)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,window,pool,keep", [(64, 100, 4, 0), (128, 300, 16, 0), (64, 128, 1, 0), (40, 33, 0, 20), (160, 64, 0, 3)])
@pytest.mark.parametrize("lens", [[5, 400, 129], [1000], [210] * 20])
def test_windows(dt, D, window, pool, keep, lens):
    _check(dt, lens, 8, 2, D, D, lambda q, k, v, kb, vb, m, on: S.window_pool_attention(
        q, None, k, v, kb, vb, m, D ** -0.5, window, pool or None, None, keep), pool=pool)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("chunk,cap,slopes", [(None, 5.0, False), (64, None, True), (50, 2.0, True)])
@pytest.mark.parametrize("lens", [[1, 50, 51, 200], [130] * 18])
def test_chunks(dt, chunk, cap, slopes, lens):
    gate = torch.randn(len(lens), 8 * 64, generator=torch.Generator().manual_seed(2)).to(dt)
    sl = S.distance_slopes(8) if slopes else None
    _check(dt, lens, 8, 2, 64, 64, lambda q, k, v, kb, vb, m, on: S.chunk_attention(
        q, on(gate), k, m, 0.125, chunk, cap, on(sl), on(torch.zeros(8))), latent=True)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_splits_bias_and_view(dt):
    """More keys than one workgroup walks, a bias by distance, a result written times a number into a wider matrix."""
    rel = torch.randn(8, 70, generator=torch.Generator().manual_seed(3))

    def run(q, k, v, kb, vb, m, on):
        wide = torch.zeros(q.shape[0], 8 * 96 + 32, dtype=q.dtype, device=q.device)
        S.window_pool_attention(q, None, k, v, None, None, m, 0.1, None, None, None, 0, on(rel), wide[:, 32:], 0.5)
        assert (wide[:, :32] == 0).all()
        return wide
    _check(dt, [3000, 1, 1700], 8, 2, 96, 96, run)


@pytest.mark.parametrize("dt,H,G,D,Dv,lens", [
    (torch.bfloat16, 16, 1, 320, 256, [2600, 900, 2599, 1] * 2),   # four heads a workgroup, split
    (torch.bfloat16, 8, 8, 64, 64, [2100]),                         # one head, split
    (torch.bfloat16, 16, 4, 64, 64, [1600] * 17),                   # more than 256 heads, split
    (torch.float32, 16, 4, 128, 128, [2000, 3]),                    # one head, split
    (torch.float32, 16, 1, 160, 128, [1300] * 12),                  # the general kernel's, split
    (torch.float32, 12, 3, 64, 64, [70] * 30),                      # four heads a workgroup, whole
    (torch.float32, 12, 3, 64, 192, [70] * 30),                     # the same with the widest values
    (torch.float32, 32, 8, 64, 64, [20] * 150)])                    # the general kernel's, 1200 workgroups, three to a CU
def test_every_form_of_the_plan(dt, H, G, D, Dv, lens):
    _check(dt, lens, H, G, D, Dv, lambda q, k, v, kb, vb, m, on: S.window_pool_attention(
        q, None, k, v, None, None, m, D ** -0.5, None, None), latent=G == 1)


def test_scores_of_minus_infinity_and_page_sizes():
    """A key whose score is -inf has no weight; pages that are no power of two stay with the general kernel."""
    for page in (16, 24):
        k = torch.randn(4, page, 1, 64, device="cuda")
        k[0, 3] = -float("inf")
        q = torch.rand(1, 4, 64, device="cuda") + 0.1
        table = torch.arange(4, device="cuda", dtype=torch.int32).view(1, 4)
        v = torch.randn_like(k)
        m = S.RaggedMeta.build([(0, 59, 1)], table, page, "cuda")
        got = S.window_pool_attention(q, None, k, v, None, None, m, 0.1, None, None)
        s = torch.einsum("hd,jd->hj", q[0].double(), k.view(-1, 64)[:60].double()) * 0.1
        assert s[:, 3].isneginf().all()
        ref = (torch.softmax(s, -1) @ v.view(-1, 64)[:60].double()).view(1, -1)
        assert (got.double() - ref).abs().max() < 1e-5


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,D,R,vdim", [(4, 320, 256, 128), (16, 288, 256, 64), (5, 160, 128, 64), (3, 72, 64, 128), (2, 200, 136, 64),
                                        (4, 64, 48, 40)])
@pytest.mark.parametrize("lens", [[1], [127, 300, 16, 129], [2000, 3]])
@pytest.mark.parametrize("gated", [False, True])
def test_latent_heads(dt, H, D, R, vdim, lens, gated):
    """Each head's result times its matrix: columns and ranks beside the thread layout, keys split, other columns than the fused ones."""
    g = torch.Generator().manual_seed(4)
    uv = (torch.randn(H, R, vdim, generator=g) * R ** -0.5).to(dt)
    wide = torch.randn(len(lens), 24 + H * vdim, generator=g).to(dt)
    sink = torch.linspace(-1, 3, H)
    table = torch.randperm(len(lens) * 125, generator=g).view(len(lens), 125).int()
    lat = torch.randn(len(lens) * 125, PAGE, 1, D, generator=g).to(dt)
    q = torch.randn(len(lens), H, D, generator=g).to(dt)

    def on(dev, f):
        c = lambda t: t.to(dev).to(f)
        return S.latent_attention(c(q), c(lat), c(uv), c(wide)[:, 24:] if gated else None, _meta(lens, dev, table), D ** -0.5, 100,
                                  sink.to(dev))
    got, ref = on("cuda", dt).float().cpu(), on("cpu", torch.float32)
    # one rounding of the result and, where the launches are two, one of each of the R numbers behind it (weights of norm about 1)
    eps = 2.0 ** -6 if dt == torch.bfloat16 else 2.0 ** -16
    assert torch.isfinite(got).all() and ((got - ref).abs() <= eps * (1 + ref.abs())).all(), (got - ref).abs().max()
