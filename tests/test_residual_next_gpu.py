"""A sublayer's residual sum with the next sublayer's row in one launch (residual_next.hip) against the two ops in fp32 on the
CPU, at the edges of a thread's runs of four and at widths and group sizes that stay with the separate kernels; and whole models
with every layer watched (the separate calls) and unwatched."""
import pytest
import torch

import edgellm.ops.seqmix as S

pytestmark = pytest.mark.gpu
DT = [torch.bfloat16, torch.float32]


def _rand(g, *s):
    return torch.randn(*s, generator=g)


def _near(got, ref, dt):
    # fp32 sums of up to 4096 terms in another order (1e-5 of the row's size of about 10), one rounding to dt
    assert ((got.float().cpu() - ref.float()).abs() <= 1e-4 + (2.0 ** -7 if dt == torch.bfloat16 else 1e-5) * ref.float().abs()).all()


def _results(g, T, K, W, dt, with_y, with_w=True):
    y = _rand(g, T, W).to(dt) if with_y else None
    parts = _rand(g, T, K, W).to(dt) if K else None
    return y, parts, _rand(g, T, K) if K and with_w else None


cuda = lambda t: None if t is None else t.cuda()
cpu = lambda t: None if t is None else (t.float() if t.is_floating_point() else t)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("W", [64, 256, 1020, 1024, 1028, 2048, 4096, 4100, 1022])
@pytest.mark.parametrize("T,K,with_y", [(1, 0, True), (5, 3, True), (4, 5, False)])
def test_layer_norm_then_taps(dt, W, T, K, with_y):
    g = torch.Generator().manual_seed(W + K)
    x, w, b, cw, state = _rand(g, T, W), _rand(g, W), _rand(g, W), _rand(g, W, 4), _rand(g, T + 2, 3, W)
    y, parts, pw = _results(g, T, K, W, dt, with_y)
    seqs = [(s, (0, 1, 2, 3, 9)[i % 5], 1) for i, s in enumerate(torch.randperm(T + 2, generator=g)[:T].tolist())]
    for s, p, _ in seqs:
        if p:
            state[s, :max(0, 3 - p)] = 0                    # a tail has nothing before position 0
    table = torch.zeros(T + 2, 1, dtype=torch.int32)
    out = {}
    for dev in ("cuda", "cpu"):
        m = S.RaggedMeta.build(seqs, table.to(dev), 16, dev)
        put = cuda if dev == "cuda" else cpu
        xs, st = x.to(dev, copy=True), state.to(dev, copy=True)
        h = S.layer_norm_residual_canon(xs, put(y), put(w), put(b), 1e-6, put(parts), put(pw), put(cw), st, m, dt if dev == "cuda" else torch.float32)
        out[dev] = (xs, st, h)
    assert out["cuda"][2].dtype == dt
    _near(out["cuda"][0], out["cpu"][0], torch.float32)
    _near(out["cuda"][1], out["cpu"][1], torch.float32)
    _near(out["cuda"][2], out["cpu"][2], dt)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("W", [64, 256, 1020, 1028, 2048, 4096, 4100, 1022])
@pytest.mark.parametrize("T,K,with_y", [(1, 0, True), (5, 3, True), (4, 5, False)])
def test_layer_norm_then_layer_norm(dt, W, T, K, with_y):
    g = torch.Generator().manual_seed(W + K)
    x, w, b, w2, b2 = _rand(g, T, W), _rand(g, W), _rand(g, W), _rand(g, W), _rand(g, W)
    y, parts, pw = _results(g, T, K, W, dt, with_y)
    a, xa = x.cuda(), x.clone()
    h = S.layer_norm_residual_norm(a, cuda(y), cuda(w), cuda(b), 1e-6, cuda(parts), cuda(pw), cuda(w2), cuda(b2), 1e-5, dt)
    ref = S.layer_norm_residual_norm(xa, cpu(y), w, b, 1e-6, cpu(parts), pw, w2, b2, 1e-5, torch.float32)
    _near(a, xa, torch.float32)
    _near(h, ref, dt)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("W,groups,groups2", [(256, 1, 1), (1024, 4, 2), (1280, 1, 5), (2048, 2, 8), (2304, 3, 1), (4096, 16, 1), (1024, 8, 2), (96, 2, 3),
                                              (4352, 1, 17)])
@pytest.mark.parametrize("T,K,with_y,with_w", [(1, 0, True, True), (7, 3, False, False), (3, 5, True, True)])
def test_group_norm_then_group_norm(dt, W, groups, groups2, T, K, with_y, with_w):
    g = torch.Generator().manual_seed(W + K)
    x, w, w2 = _rand(g, T, W), _rand(g, W), _rand(g, W)
    y, parts, pw = _results(g, T, K, W, dt, with_y, with_w)
    a, xa = x.cuda(), x.clone()
    h = S.group_norm_residual_norm(a, cuda(y), cuda(w), groups, 1e-6, 0.3, cuda(parts), cuda(pw), cuda(w2), groups2, 1e-5, dt)
    ref = S.group_norm_residual_norm(xa, cpu(y), w, groups, 1e-6, 0.3, cpu(parts), pw, w2, groups2, 1e-5, torch.float32)
    _near(a, xa, torch.float32)
    _near(h, ref, dt)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("T,W", [(512, 2304), (513, 2304), (513, 2048)])
def test_group_norms_of_many_rows(dt, T, W):
    """Both sides of the line from which long rows run two launches."""
    g = torch.Generator().manual_seed(T)
    x, w, w2 = _rand(g, T, W), _rand(g, W), _rand(g, W)
    y, parts, pw = _results(g, T, 2, W, dt, True, True)
    a, xa = x.cuda(), x.clone()
    h = S.group_norm_residual_norm(a, cuda(y), cuda(w), 1, 1e-6, 0.3, cuda(parts), cuda(pw), cuda(w2), 1, 1e-5, dt)
    ref = S.group_norm_residual_norm(xa, cpu(y), w, 1, 1e-6, 0.3, cpu(parts), pw, w2, 1, 1e-5, torch.float32)
    _near(a, xa, torch.float32)
    _near(h, ref, dt)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("W", [64, 256, 1020, 1024, 2052, 4096, 4100, 1022])
@pytest.mark.parametrize("T,extra", [(1, True), (6, False)])
def test_combine_then_norm(dt, W, T, extra):
    g = torch.Generator().manual_seed(W)
    x, wl, wr, gain = _rand(g, T, W), _rand(g, W), _rand(g, W), _rand(g, 1)
    l, r, e = _rand(g, T, W).to(dt), _rand(g, T, W).to(dt), _rand(g, T, W).to(dt) if extra else None
    a, xa = x.cuda(), x.clone()
    h = S.combine_residual_norm(a, cuda(l), cuda(r), cuda(wl), cuda(wr), 1e-6, cuda(e), cuda(gain), 1e-5, dt)
    ref = S.combine_residual_norm(xa, cpu(l), cpu(r), wl, wr, 1e-6, cpu(e), gain, 1e-5, torch.float32)
    _near(a, xa, torch.float32)
    _near(h, ref, dt)


@pytest.mark.parametrize("family", ["nudadra", "pagonex", "vetevik"])
@pytest.mark.parametrize("loop", [None, "project", "add_embed", "plain"])
def test_watched_layers_give_the_same_logits(family, loop):
    """A hook on a layer keeps its input a call of its own; both forms read the same stream, through looped spans too."""
    from edgellm.engine import ragged_bench as rb
    from edgellm.engine.ragged import RaggedEngine
    from edgellm.models.configs import LoopSpec
    from edgellm.models.hybrid import HybridLM
    size = {"nudadra": rb.SIZES, "pagonex": rb.PAGONEX_SIZES, "vetevik": rb.VETEVIK_SIZES}[family]["w1024"]
    make = {"nudadra": rb.hybrid_config, "pagonex": rb.pagonex_config, "vetevik": rb.vetevik_config}[family]
    cfg = make(dict(size, layers=4, vocab=128))
    cfg = cfg.replace(loop=LoopSpec(1, 3, 2, loop) if loop else None)
    torch.manual_seed(0)
    model = HybridLM(cfg, torch.float32, "cuda")
    for p in model.parameters():
        if p.dim() > 1:
            p.data.normal_(0, 0.02)
    res = []
    for watched in (False, True):
        hooks = [m.register_forward_hook(lambda *a: None) for m in model.modules() if m is not model] if watched else []
        eng = RaggedEngine(model, 256, slots=2, page=16, use_graphs=not watched)     # (captured steps want every row)
        out = [eng.step([(0, list(range(5, 25)), [19]), (1, [7, 9], [1])])]
        for t in range(4):
            out.append(eng.step([(0, [t + 1], [0]), (1, [t + 3], [0])]))
        res.append(torch.cat(out))
        for h in hooks:
            h.remove()
    assert res[0].std() > 0
    assert (res[0] - res[1]).abs().max() <= 1e-4 * res[1].abs().max()
