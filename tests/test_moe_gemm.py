"""The grouped expert kernels of prompt-sized steps (csrc/seqmix/moe_gemm.hip) against the float64 form of the same
experts, at the edges of their tiles and of the routing."""
import pytest
import torch

import edgellm  # noqa: F401
from edgellm.ops import seqmix

gpu = pytest.mark.gpu


def reference(h, idx, w_gu, w_down, act, limit, in_w):
    T, top = idx.shape
    out = torch.zeros(T, top, w_down.shape[1], dtype=torch.float64)
    h, w_gu, w_down = (t.cpu().double() for t in (h, w_gu, w_down))
    idx = idx.cpu().long()
    ff = w_down.shape[2]
    for e in idx.unique().tolist():
        t, k = (idx == e).nonzero(as_tuple=True)
        u = h[t] @ w_gu[e].T
        if act == "relu2":
            y = torch.relu(u) ** 2
        elif act == "silu_glu":
            u = u if in_w is None else u * in_w.cpu().double()[t, k][:, None]
            y = torch.nn.functional.silu(u[:, :ff]) * u[:, ff:]
        else:
            g, up = u[:, :ff].clamp(max=limit), u[:, ff:].clamp(-limit, limit)
            y = g * torch.sigmoid(1.702 * g) * (up + 1)
        out[t, k] = y @ w_down[e].T
    return out


def inputs(T, top, E, W, ff, act, seed=0):
    g = torch.Generator().manual_seed(seed)
    up = 1 if act == "relu2" else 2
    h = torch.randn(T, W, generator=g).bfloat16()
    w_gu = (torch.randn(E, up * ff, W, generator=g) * W ** -0.5).bfloat16()
    w_down = (torch.randn(E, W, ff, generator=g) * ff ** -0.5).bfloat16()
    idx = torch.rand(T, E, generator=g).topk(top, -1).indices.int()
    in_w = torch.rand(T, top, generator=g) if act == "silu_glu" else None
    return [t.cuda() if t is not None else None for t in (h, idx, w_gu, w_down, in_w)]


# the hidden unit is stored in bf16 (relative rounding 2^-9 per term, random) and so is the result: 2-norm error about
# 2^-9 sqrt(2 / 3) each = 2.3e-3 together; twice that is the bound
TOL = 5e-3


@pytest.fixture
def every_size(monkeypatch):
    """Small experts too, which steps below MOE_GEMM_MIN tokens otherwise run by rows."""
    monkeypatch.setattr(seqmix, "MOE_MFMA_WORK", 0)


@gpu
@pytest.mark.parametrize("act", ["glu_clamp", "silu_glu", "relu2"])
@pytest.mark.parametrize("T,top,E,W,ff", [
    (10, 2, 5, 64, 64),          # one k step, fewer rows than experts can fill
    (33, 3, 4, 128, 192),        # rows per expert about one 32-row tile; columns past a whole 128
    (100, 1, 2, 192, 64),        # 64-row tiles with a remainder
    (257, 2, 3, 256, 320),       # 128-row tiles with a remainder
    (1030, 4, 16, 320, 128),     # several tiles per expert
    (70, 1, 512, 64, 128)])      # the most experts
def test_grouped_experts_against_float64(T, top, E, W, ff, act, every_size):
    h, idx, w_gu, w_down, in_w = inputs(T, top, E, W, ff, act)
    assert seqmix.moe_grouped(h, idx, w_gu, w_down, act, in_w)
    got = seqmix.moe_experts(h, idx, w_gu, w_down, 1.5, act, in_w).cpu().double()
    want = reference(h, idx, w_gu, w_down, act, 1.5, in_w)
    assert ((got - want).norm() / want.norm()) < TOL
    assert ((got - want).norm(dim=-1) / want.norm(dim=-1).clamp_min(1e-3)).max() < 4 * TOL


@gpu
@pytest.mark.parametrize("T,top,E,W,ff,act", [
    (400, 2, 8, 64, 1024, "glu_clamp"),          # 128-row tiles: one k step in the first product
    (400, 2, 8, 1024, 64, "silu_glu"),           # one in the second
    (400, 2, 8, 64, 1024, "relu2"),
    (3840, 3, 48, 1024, 192, "glu_clamp"),       # three in the second, every stage of the weights' ring once; the first one's rings are equal
    (3840, 3, 48, 192, 1024, "relu2"),           # three in the first; equal rings in the second
    (2400, 2, 8, 1024, 1024, "glu_clamp"),       # unequal, then equal
    (1600, 2, 16, 512, 1024, "silu_glu"),        # equal, then unequal
    (4688, 1, 8, 256, 3072, "relu2"),
    (3200, 2, 32, 1024, 1024, "silu_glu"),       # 256-row tiles, gated, spread starts: equal rings
    (3840, 2, 32, 1024, 1024, "relu2"),          # squared units
    (2960, 2, 8, 1536, 1024, "glu_clamp")])      # and starts in step
def test_rings_of_unequal_depth_against_float64(T, top, E, W, ff, act):
    h, idx, w_gu, w_down, in_w = inputs(T, top, E, W, ff, act, T)
    assert seqmix.moe_grouped(h, idx, w_gu, w_down, act, in_w)
    got = seqmix.moe_experts(h, idx, w_gu, w_down, 1.5, act, in_w).cpu().double()
    want = reference(h, idx, w_gu, w_down, act, 1.5, in_w)
    assert ((got - want).norm(dim=-1) / want.norm(dim=-1).clamp_min(1e-3)).max() < 4 * TOL


@gpu
def test_small_experts_of_small_steps_run_by_rows():
    """Pairs times an expert's numbers on both sides of MOE_MFMA_WORK, and a step of MOE_GEMM_MIN tokens: the same result."""
    for T, W, ff, grouped in ((12, 256, 128, False), (42, 256, 128, False), (43, 256, 128, True), (64, 64, 64, True), (63, 64, 64, False)):
        h, idx, w_gu, w_down, in_w = inputs(T, 2, 8, W, ff, "silu_glu", T)
        assert seqmix.moe_grouped(h, idx, w_gu, w_down, "silu_glu", in_w) == grouped
        got = seqmix.moe_experts(h, idx, w_gu, w_down, 0.0, "silu_glu", in_w).cpu().double()
        want = reference(h, idx, w_gu, w_down, "silu_glu", 0.0, in_w)
        assert (got - want).norm() < TOL * want.norm()


@gpu
@pytest.mark.parametrize("T,W,ff,sff", [(9, 1024, 512, 1024), (10, 1024, 512, 1024), (33, 512, 1024, 512), (63, 1024, 512, 576),
                                        (12, 1024, 512, 1032), (40, 256, 128, 192)])
def test_shared_expert_of_small_steps_squares_in_fp32(T, W, ff, sff):
    """Steps below MOE_GEMM_MIN tokens: u is squared before it is rounded.  The unit and the result are rounded to bf16 (rms
    2^-9 each at most, random): 2.8e-3 together; a u rounded first would add 2 x 1.6e-3 to the unit (4e-3 measured)."""
    from edgellm.models.configs import MoESpec
    from edgellm.models.moe import MoEFeedForward
    g = torch.Generator().manual_seed(T)
    m = MoEFeedForward(MoESpec(8, 3, 1.0, ff, shared_ff=sff, router="softmax", act="relu2", correction=True, groups=4, groups_keep=2,
                               shared_gate=True), W, torch.bfloat16, torch.device("cuda:0"))
    for p in m.parameters():
        p.data.copy_(torch.randn(p.shape, generator=g) * p.shape[-1] ** -0.5)
    h = torch.randn(T, W, generator=g).bfloat16().cuda()
    f = m.run(h)
    d = lambda t: t.cpu().double()
    want = torch.relu(d(h) @ d(m.shared_gu.weight).T) ** 2 @ d(m.shared_down.weight).T
    assert (d(f.shared) - want).norm() < 2.8e-3 * want.norm()
    idx = seqmix.moe_route_grouped(h, m.router, 3, 1.0, m.correction, 4, 2, True)[0]
    want = reference(h, idx, m.w_gu, m.w_down, "relu2", 0.0, None)
    assert f.rows is None and (d(f.parts) - want).norm() < 2.8e-3 * want.norm()


@gpu
@pytest.mark.parametrize("case", ["one expert", "first and last", "idle neighbours"])
def test_grouped_experts_with_skewed_routing(case):
    T, E = 300, 9
    h, idx, w_gu, w_down, _ = inputs(T, 2, E, 64, 128, "relu2", 3)
    if case == "one expert":
        idx.fill_(4)
    elif case == "first and last":
        idx[:, 0], idx[:, 1] = 0, E - 1
    else:
        idx[:, 0], idx[:, 1] = 2, 7
    got, rows = seqmix.moe_experts(h, idx, w_gu, w_down, 0.0, "relu2", sorted_rows=True)
    assert rows is None
    want = reference(h, idx, w_gu, w_down, "relu2", 0.0, None)
    assert ((got.cpu().double() - want).norm() / want.norm()) < TOL


@gpu
def test_grouped_experts_keep_nan_and_infinity_in_their_rows():
    h, idx, w_gu, w_down, in_w = inputs(64, 2, 4, 128, 64, "silu_glu", 5)
    clean = seqmix.moe_experts(h, idx, w_gu, w_down, 0.0, "silu_glu", in_w)
    bad = h.clone()
    bad[7], bad[40, 3] = float("nan"), float("inf")
    got = seqmix.moe_experts(bad, idx, w_gu, w_down, 0.0, "silu_glu", in_w)
    keep = torch.ones(64, dtype=torch.bool)
    keep[[7, 40]] = False
    assert torch.equal(got[keep.cuda()], clean[keep.cuda()])
    assert got[7].isnan().all()


@gpu
def test_steps_that_the_grouped_kernels_do_not_take():
    h, idx, w_gu, w_down, in_w = inputs(80, 2, 4, 128, 96, "silu_glu", 6)          # ff is no whole 64
    assert not seqmix.moe_grouped(h, idx, w_gu, w_down, "silu_glu", in_w)
    got = seqmix.moe_experts(h, idx, w_gu, w_down, 0.0, "silu_glu", in_w).cpu().double()
    want = reference(h, idx, w_gu, w_down, "silu_glu", 0.0, in_w)
    assert ((got - want).norm() / want.norm()) < 2 * TOL                            # both halves rounded to bf16 as well
    h, idx, w_gu, w_down, in_w = inputs(80, 2, 4, 128, 64, "silu_glu", 7)
    wide = torch.randn(80, 256, device="cuda").bfloat16()
    wide[:, :128] = h
    assert not seqmix.moe_grouped(wide[:, :128], idx, w_gu, w_down, "silu_glu", in_w)   # rows of a wider tensor
    assert not seqmix.moe_grouped(h.float(), idx, w_gu.float(), w_down.float(), "silu_glu", in_w)
    assert not seqmix.moe_grouped(h[:5], idx[:5], w_gu, w_down, "silu_glu", in_w[:5])
    assert torch.allclose(seqmix.moe_experts(wide[:, :128], idx, w_gu, w_down, 0.0, "silu_glu", in_w).float(),
                          seqmix.moe_experts(h, idx, w_gu, w_down, 0.0, "silu_glu", in_w).float(), atol=3e-2, rtol=3e-2)


@gpu
@pytest.mark.parametrize("E,W,ff,T,top", [(32, 1024, 2048, 400, 4), (32, 1024, 2048, 401, 4), (32, 1024, 1984, 401, 4), (4, 64, 64, 256, 2),
                                          (4, 64, 64, 257, 2), (32, 1024, 2048, 488, 4), (32, 1024, 2048, 492, 4)])
def test_lines_between_tile_heights(E, W, ff, T, top, every_size):
    """Rows per expert around 50, 60 and 128: 488 tokens run 64-row tiles by estimate, 492 run 128-row ones."""
    g = torch.Generator(device="cuda").manual_seed(T + ff)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    h, w_gu, w_down = r(T, W).bfloat16(), (r(E, ff, W) * W ** -0.5).bfloat16(), (r(E, W, ff) * ff ** -0.5).bfloat16()
    idx = torch.rand(T, E, generator=g, device="cuda").topk(top, 1)[1].int()
    assert seqmix.moe_grouped(h, idx, w_gu, w_down, "relu2", None)
    got = seqmix.moe_experts(h, idx, w_gu, w_down, 0.0, "relu2")
    for e in range(E):
        t, k = (idx == e).nonzero(as_tuple=True)
        want = torch.relu(h[t].double() @ w_gu[e].double().t()) ** 2 @ w_down[e].double().t()
        assert (got[t, k].double() - want).norm() < TOL * want.norm()


@gpu
@pytest.mark.parametrize("act,T,top,E,W,ff", [("glu_clamp", 5200, 3, 7, 960, 1088), ("silu_glu", 5200, 3, 7, 960, 1088),
                                              ("relu2", 10200, 2, 5, 2048, 2048), ("glu_clamp", 4600, 3, 7, 960, 1088),
                                              ("silu_glu", 4600, 3, 7, 960, 1088)])
def test_tall_tiles(act, T, top, E, W, ff):
    """Sizes whose estimates choose 256 x 256 tiles (10200 and 4600 tokens) or nearly do, with remainders of rows and columns (960 = 3 x 256
    + 192)."""
    g = torch.Generator(device="cuda").manual_seed(T)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    h, w_gu = r(T, W).bfloat16(), (r(E, ff if act == "relu2" else 2 * ff, W) * W ** -0.5).bfloat16()
    w_down, in_w = (r(E, W, ff) * ff ** -0.5).bfloat16(), torch.rand(T, top, generator=g, device="cuda") if act == "silu_glu" else None
    idx = torch.rand(T, E, generator=g, device="cuda").topk(top, 1)[1].int()
    assert seqmix.moe_grouped(h, idx, w_gu, w_down, act, in_w)
    got = seqmix.moe_experts(h, idx, w_gu, w_down, 1.5, act, in_w)
    err = norm = 0.0
    for e in range(E):
        t, k = (idx == e).nonzero(as_tuple=True)
        u = h[t].double() @ w_gu[e].double().t()
        gate, up = u[:, :ff], u[:, ff:]
        if act == "relu2":
            y = torch.relu(u) ** 2
        elif act == "glu_clamp":
            gate = gate.clamp(max=1.5)
            y = gate * torch.sigmoid(1.702 * gate) * (up.clamp(-1.5, 1.5) + 1)
        else:
            rw = in_w[t, k].double()[:, None]
            y = torch.nn.functional.silu(rw * gate) * (rw * up)
        want = y @ w_down[e].double().t()
        d = got[t, k].double() - want
        assert (d.norm(dim=-1) / want.norm(dim=-1).clamp_min(1e-3)).max() < 4 * TOL
        err, norm = err + d.norm().item() ** 2, norm + want.norm().item() ** 2
    assert err ** 0.5 < TOL * norm ** 0.5
