"""The last block's sum and the final LayerNorm in the LM head's launch, and fp16 scores read by the sampler as they are."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,V,top_k,top_p,do_sample", [
    (1, 50304, 50, 0.9, True),       # 16-byte loads, chunks
    (3, 1003, 40, 0.95, True),       # no whole 8: element by element
    (130, 2048, 20, 0.9, True),      # a row a workgroup
    (2, 4096, 200, 1.0, True),       # more than a chunk's candidates
    (2, 5000, 0, 1.0, True),         # the whole row
    (4, 777, 0, 1.0, False)])        # greedy
@pytest.mark.parametrize("form", ["rows", "gaps", "off 16 bytes"])
def test_fp16_scores_draw_what_their_fp32_values_do(cuda, B, V, top_k, top_p, do_sample, form):
    from edgellm import ops
    g = torch.Generator().manual_seed(V)
    x = (torch.randn(B, V, generator=g) * 4).half().cuda()
    if form == "gaps":
        wide = torch.zeros(B, V + 8, dtype=torch.float16, device="cuda")
        wide[:, :V] = x
        x = wide[:, :V]
    elif form == "off 16 bytes":
        x = torch.cat([torch.zeros(1, dtype=torch.float16, device="cuda"), x.flatten()])[1:].view(B, V)
    seen = (torch.rand(B, V, generator=g) < 0.1).byte().cuda()
    seen2 = seen.clone()
    rng = torch.tensor([7, 3], dtype=torch.int32, device="cuda")
    a = ops.sample(x, seen, 0.7, top_k, top_p, 1.2, rng, do_sample)
    b = ops.sample(x.float().contiguous(), seen2, 0.7, top_k, top_p, 1.2, rng, do_sample)
    assert torch.equal(a, b) and torch.equal(seen, seen2)      # widening is exact


@pytest.mark.parametrize("top_k", [128, 129, 1000])            # the last two: widened in front of a row's many passes
def test_fp16_scores_of_a_decode_step(cuda, top_k):
    """The sampler with the step's bookkeeping behind it, eager and in a graph."""
    from edgellm import ops
    B, V = 3, 4096
    x = (torch.randn(B, V, generator=torch.Generator().manual_seed(top_k)) * 4).half().cuda()

    def state():
        z = lambda n, t: torch.zeros(n, dtype=t, device="cuda")
        return dict(seen=z((B, V), torch.uint8), rng=torch.tensor([5, 0], dtype=torch.int32, device="cuda"), tok=z(B, torch.long),
                    out=z((B, 8), torch.long), step=z(1, torch.long), pos=z(B, torch.int32), lens=z(B, torch.int32), ctr=z(1, torch.int32))

    def step(s, lg):
        return ops.sample_advance(lg, s["seen"], 0.8, top_k, 0.95, 1.1, s["rng"], s["tok"], s["out"], s["step"], s["pos"], s["lens"], s["ctr"])
    a, b, c, wide = state(), state(), state(), x.float()
    for _ in range(4):
        assert torch.equal(step(a, x), step(b, wide))
    g = torch.cuda.CUDAGraph()
    step(state(), x)
    with torch.cuda.graph(g):
        step(c, x)
    for _ in range(4):
        g.replay()
    for k in a:
        assert torch.equal(a[k], b[k]) and torch.equal(a[k], c[k]), k


@pytest.mark.parametrize("family,dtype", [("gpt_neox", torch.float16), ("phi", torch.bfloat16)])
@pytest.mark.parametrize("rows", [1, 4])
def test_head_takes_both_branches(cuda, family, dtype, rows, monkeypatch):
    from edgellm.models import build_model, tiny
    from edgellm.models.layers import BranchRows, Linear
    cfg = tiny(family, num_layers=1, hidden_size=256, num_heads=4, num_kv_heads=4, intermediate_size=512, rotary_dim=32)
    model = build_model(cfg, dtype=dtype, device="cuda", seed=3)
    g = torch.Generator().manual_seed(rows)
    a, m, r = (torch.randn(rows, 256, generator=g).to(dtype).cuda() for _ in range(3))
    took = []
    real = Linear.forward_ln
    monkeypatch.setattr(Linear, "forward_ln", lambda self, x, *k: took.append(1) or real(self, x, *k))

    class Ctx:
        T = 1
    got = model.head(BranchRows(a, m), r, Ctx)
    assert took
    want = model.head(m + a, r, Ctx)
    assert len(took) == 1
    eps = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    # the same normalised rows; fp32 sums that meet in another order, so at most the last rounding differs
    h = torch.nn.functional.layer_norm((m + a).float() + r.float(), (256,)).abs() @ model.lm_head.weight.float().abs().T
    assert ((got.float() - want.float()).abs() <= 2 * eps * want.float().abs() + 2.0 ** -22 * 256 ** 0.5 * h + 1e-6).all()
    seen = []
    hook = model.final_norm.register_forward_hook(lambda mod, i, o: seen.append(1))
    assert torch.equal(model.head(BranchRows(a, m), r, Ctx), want) and seen and len(took) == 1     # a watched norm is called
    hook.remove()
