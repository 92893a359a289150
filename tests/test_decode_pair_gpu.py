"""Independent parts of a parallel-residual decode step in one launch (decode_pair.hip) against float64 and the separate ops."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _rows(g, *shape, dtype, scale=1.0):
    return (torch.randn(*shape, generator=g) * scale).to(dtype).cuda()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,Ko,Kd", [(1, 16, 64, 64), (2, 2048, 2048, 8192), (4, 2560, 2560, 10240), (3, 48, 320, 192), (1, 272, 2112, 512)])
def test_o_down(cuda, dtype, M, N, Ko, Kd):
    from edgellm import ops
    g = torch.Generator().manual_seed(N + Ko + Kd + M)
    for with_bias in (False, True):
        xs, ws, bs = [], [], []
        for K in (Ko, Kd):
            xs.append(_rows(g, M, K, dtype=dtype))
            ws.append(_rows(g, N, K, dtype=dtype, scale=K ** -0.5))
            bs.append(_rows(g, N, dtype=dtype) if with_bias else None)
        out = ops.ext().decode_o_down(xs[0], ops.pack_bf16_weight(ws[0]), bs[0], xs[1], ops.pack_bf16_weight(ws[1]), bs[1], N)
        for y, x, w, b, K in zip(out, xs, ws, bs, (Ko, Kd)):
            ref = x.double() @ w.double().T + (0 if b is None else b.double())
            # one rounding of the result and fp32 sums of K products
            bound = EPS[dtype] * ref.abs() + 2.0 ** -24 * K * (x.double().abs() @ w.double().abs().T)
            assert ((y.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("act", ["gelu", "gelu_tanh"])
@pytest.mark.parametrize("B,D,Hq,Hkv,S,lens,N,K", [
    (1, 256, 8, 8, 128, [1], 8192, 2048), (1, 80, 32, 32, 320, [300], 10240, 2560), (4, 64, 12, 12, 700, [3, 700, 257, 64], 64, 768),
    (2, 128, 8, 2, 256, [255, 256], 16, 64), (3, 256, 4, 1, 1100, [1100, 900, 5], 400, 320)])
def test_attn_up(cuda, dtype, act, B, D, Hq, Hkv, S, lens, N, K):
    from edgellm import ops
    g = torch.Generator().manual_seed(B * D + S + N)
    rot = 16 * (D // 32)
    qkv = _rows(g, B, (Hq + 2 * Hkv) * D, dtype=dtype)
    k1, v1 = (_rows(g, B, Hkv, S, D, dtype=dtype) for _ in range(2))
    k2, v2 = k1.clone(), v1.clone()
    seq = torch.tensor(lens, dtype=torch.int32).cuda()
    pos = seq - 1
    rope = ops.rope_tables(rot, S, 10000.0, None, device="cuda")
    y, w, b = _rows(g, B, K, dtype=dtype), _rows(g, N, K, dtype=dtype, scale=K ** -0.5), _rows(g, N, dtype=dtype)
    ref, _ = ops.decode_attention_fused(qkv, pos, rope, k1, v1, seq, Hq, D ** -0.5, max(lens), rot)
    a, h = ops.decode_attn_up(qkv, pos, rope, k2, v2, seq, Hq, D ** -0.5, max(lens), rot, y, ops.pack_bf16_weight(w), b, N, act)
    assert torch.equal(k1, k2) and torch.equal(v1, v2)
    # the same products and weights; the fp32 sums meet in another order: at most the last rounding differs
    assert ((a.view(B, Hq, D).float() - ref.float()).abs() <= 2 * EPS[dtype] * ref.float().abs() + 1e-5).all()
    z = y.double() @ w.double().T + b.double()
    e = EPS[dtype] * z.abs() + 2.0 ** -24 * K * (y.double().abs() @ w.double().abs().T)
    gelu = lambda t: torch.nn.functional.gelu(t, approximate="tanh" if act == "gelu_tanh" else "none")  # noqa: E731
    # gelu's slope is at most 1.13; then the result's own rounding and fp32 function error
    assert ((h.double() - gelu(z)).abs() <= 1.13 * e + EPS[dtype] * gelu(z).abs() + 2.0 ** -22 * (1 + z.abs())).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K", [(1, 2048), (4, 2560), (3, 768)])
@pytest.mark.parametrize("two", [False, True])
def test_norm_of_both_branches_is_the_norm_kernels(cuda, dtype, M, K, two):
    from edgellm import ops
    g = torch.Generator().manual_seed(M * K)
    x, x2, res = (_rows(g, M, K, dtype=dtype) for _ in range(3))
    g1, b1, g2, b2 = (_rows(g, K, dtype=dtype) for _ in range(4))
    w = _rows(g, 64, K, dtype=dtype, scale=K ** -0.5)
    h, y = torch.empty_like(x), torch.empty_like(x)
    out = ops.gemv_bf16_ln(x, res, g1, b1, 1e-5, h, ops.pack_bf16_weight(w), None, 64, None, y_out=y, x2=x2,
                           gamma2=g2 if two else None, beta2=b2 if two else None)
    n1, r = ops.layer_norm(x + x2, g1, b1, 1e-5, res)
    n2, _ = ops.layer_norm(r, g2 if two else g1, b2 if two else b1, 1e-5, None)
    assert torch.equal(h, r) and torch.equal(y, n2)
    assert torch.equal(out, ops.linear_bf16(n1, w, None, packed=ops.pack_bf16_weight(w)))


@pytest.mark.parametrize("family,dtype", [("gpt_neox", torch.float16), ("phi", torch.bfloat16)])
def test_decode_steps_agree_with_the_separate_launches(cuda, family, dtype, monkeypatch):
    from edgellm.engine import Generator, SamplingParams
    from edgellm.models import build_model, tiny
    from edgellm.models.decoder import DecoderLayer
    cfg = tiny(family, num_layers=3, hidden_size=256, num_heads=4, num_kv_heads=4, intermediate_size=512, rotary_dim=32)
    model = build_model(cfg, dtype=dtype, device="cuda", seed=3)
    sp = SamplingParams(max_new_tokens=5, temperature=0.0, do_sample=False) if "do_sample" in SamplingParams.__dataclass_fields__ \
        else SamplingParams(max_new_tokens=5, top_k=1)
    prompts = [[5, 9, 2, 7, 1], [3, 8, 8, 4, 6]]
    used = []
    real = DecoderLayer._pair
    monkeypatch.setattr(DecoderLayer, "_pair", lambda self, *a: used.append(1) or real(self, *a))
    one = Generator(model, max_batch=2, max_seq=32)
    one.generate(prompts, sp, seed=1)
    k1, v1 = one.kv.k.clone(), one.kv.v.clone()
    assert used
    monkeypatch.setattr(DecoderLayer, "_pair_ok", lambda self, *a: False)
    two = Generator(model, max_batch=2, max_seq=32)
    two.generate(prompts, sp, seed=1)
    for a, b in ((k1, two.kv.k), (v1, two.kv.v)):
        d = (a.float() - b.float()).norm() / b.float().norm()
        assert d < 4 * EPS[dtype], d                     # three layers of differing last roundings
    assert math.isfinite(float(k1.float().abs().max()))


def _stepped(model, steps=2, caches=False):
    """Logits (and caches) of a two-token prompt and some decode steps of one sequence, through the model's own call."""
    from edgellm.engine import KVCache
    from edgellm.models import AttnCtx
    kv, rope = KVCache(model.cfg, 1, 16, dtype=model.dtype, device="cuda"), model.rope_table()
    at = lambda n: torch.tensor([n], dtype=torch.int32, device="cuda")
    ids = torch.tensor([[5, 9, 3, 7]], device="cuda")
    with torch.no_grad():
        out = [model(ids[:, :2], AttnCtx("prefill", 1, 2, at(0), at(2), 2, kv.rows(0, 1), rope), logits="last")]
        for t in range(steps):
            out.append(model(ids[:, 2 + t:3 + t], AttnCtx("decode", 1, 1, at(2 + t), at(3 + t), 3 + t, kv.rows(0, 1), rope)))
    return (torch.cat(out).float(), kv.k, kv.v) if caches else torch.cat(out).float()


@pytest.mark.parametrize("where", ["layer", "final_norm"])
@pytest.mark.parametrize("kind", ["hook", "pre_hook", "forward"])
def test_a_watched_layer_or_final_norm_sees_rows(cuda, where, kind, monkeypatch):
    from edgellm.models import build_model, tiny
    from edgellm.models.decoder import DecoderLayer
    cfg = tiny("gpt_neox", num_layers=4, hidden_size=256, num_heads=4, num_kv_heads=4, intermediate_size=512, rotary_dim=32)
    model, used, seen = build_model(cfg, dtype=torch.float16, device="cuda", seed=3), [], []
    real = DecoderLayer._pair
    monkeypatch.setattr(DecoderLayer, "_pair", lambda self, *a: used.append(self.idx) or real(self, *a))
    ref = _stepped(model)
    assert used == [0, 1, 2, 3] * 2
    m = model.layers[1] if where == "layer" else model.final_norm
    used.clear()
    if kind == "hook":
        h = m.register_forward_hook(lambda m, a, y: seen.append(a[:2] + y) and None)
    elif kind == "pre_hook":
        h = m.register_forward_pre_hook(lambda m, a: seen.append(a[:2]) and None)
    else:
        fwd = m.forward
        m.forward = lambda *a, **k: seen.append(a[:2]) or fwd(*a, **k)
    out = _stepped(model)
    assert len(seen) == 3 and all(isinstance(t, (torch.Tensor, type(None))) for s in seen for t in s)
    assert used == ([2, 3] if where == "layer" else [0, 1, 2]) * 2
    assert (out - ref).norm() <= 4 * EPS[torch.float16] * ref.norm()     # four layers of differing last roundings


def test_layers_that_a_program_steps_itself_give_rows(cuda):
    from edgellm.engine import KVCache
    from edgellm.models import AttnCtx, build_model, tiny
    cfg = tiny("phi", num_layers=2, hidden_size=256, num_heads=4, num_kv_heads=4, intermediate_size=512, rotary_dim=32)
    model = build_model(cfg, dtype=torch.bfloat16, device="cuda", seed=3)
    kv, at = KVCache(cfg, 1, 8, dtype=model.dtype, device="cuda"), lambda n: torch.tensor([n], dtype=torch.int32, device="cuda")
    ctx = AttnCtx("decode", 1, 1, at(0), at(1), 1, kv.rows(0, 1), model.rope_table())
    x = torch.randn(1, 256, generator=torch.Generator().manual_seed(0)).bfloat16().cuda()
    with torch.no_grad():
        a, h = model.layers[0](x, None, ctx)
        assert isinstance(a, torch.Tensor) and (a + h).shape == x.shape
        y, r = model.forward_layers(x, ctx)
    assert isinstance(y, torch.Tensor) and (y + r).shape == x.shape


@pytest.mark.parametrize("kv_heads,B,keys,together", [(2, 4, 4096, True), (2, 4, 4097, False), (4, 4, 4097, True)])
def test_long_caches_of_grouped_heads_run_apart(cuda, kv_heads, B, keys, together, monkeypatch):
    from edgellm.engine import KVCache
    from edgellm.models import AttnCtx, build_model, tiny
    from edgellm.models.decoder import DecoderLayer
    cfg = tiny("phi", num_layers=2, hidden_size=256, num_heads=4, num_kv_heads=kv_heads, intermediate_size=512, rotary_dim=32,
               max_position_embeddings=8192)
    model, used = build_model(cfg, dtype=torch.bfloat16, device="cuda", seed=3), []
    real = DecoderLayer._pair
    monkeypatch.setattr(DecoderLayer, "_pair", lambda self, *a: used.append(1) or real(self, *a))
    kv = KVCache(cfg, B, 4100, dtype=model.dtype, device="cuda")
    pos = torch.full((B,), keys - 1, dtype=torch.int32, device="cuda")
    with torch.no_grad():
        out = model(torch.ones(B, 1, dtype=torch.long, device="cuda"),
                    AttnCtx("decode", B, 1, pos, pos + 1, keys, kv.rows(0, B), model.rope_table()))
    assert bool(used) == together and torch.isfinite(out).all()


def _l8(g, N, K, bias=True):
    from edgellm.models.layers import Linear
    from edgellm.quant.linear import LLMInt8Linear
    lin = Linear(K, N, bias, torch.bfloat16, "cuda")
    lin.weight.data.copy_(torch.randn(N, K, generator=g) * K ** -0.5)
    if bias:
        lin.bias.data.copy_(torch.randn(N, generator=g))
    return LLMInt8Linear.from_float(lin)


def _row(g, K, outliers):
    x = torch.randn(1, K, generator=g)
    at = torch.randperm(K, generator=g)[:outliers]
    x[0, at] = 6.5 + 3 * torch.rand(outliers, generator=g)
    return x.to(torch.bfloat16).cuda()


@pytest.mark.parametrize("N,Ko,Kd,out", [(2560, 2560, 10240, 7), (16, 64, 4160, 0), (2048, 2048, 8192, 300), (272, 4096, 12288, 64)])
def test_llmint8_o_down_is_each_projections_own(cuda, N, Ko, Kd, out):
    from edgellm import ops
    g = torch.Generator().manual_seed(N + Kd)
    o, d = _l8(g, N, Ko), _l8(g, N, Kd, bias=False)
    x, h = _row(g, Ko, min(out, Ko)), _row(g, Kd, out)
    a, y = ops.ext().llmint8_o_down(x, *o.pair_args(), h, *d.pair_args(), N)
    assert torch.equal(a, o(x)) and torch.equal(y, d(h))


@pytest.mark.parametrize("act", ["gelu", "gelu_tanh"])
@pytest.mark.parametrize("D,Hq,Hkv,S,n,N,K", [(80, 32, 32, 128, 77, 10240, 2560), (256, 8, 8, 64, 1, 8192, 2048),
                                              (64, 4, 2, 700, 700, 48, 64), (128, 16, 16, 300, 290, 4112, 4096)])
def test_llmint8_attn_up(cuda, act, D, Hq, Hkv, S, n, N, K):
    from edgellm import ops
    g = torch.Generator().manual_seed(D + S + N)
    up = _l8(g, N, K)
    y = _row(g, K, 3)
    rot = 16 * (D // 32)
    qkv = _rows(g, 1, (Hq + 2 * Hkv) * D, dtype=torch.bfloat16)
    k1, v1 = (_rows(g, 1, Hkv, S, D, dtype=torch.bfloat16) for _ in range(2))
    k2, v2 = k1.clone(), v1.clone()
    seq = torch.tensor([n], dtype=torch.int32).cuda()
    rope = ops.rope_tables(rot, S, 10000.0, None, device="cuda")
    ref, _ = ops.decode_attention_fused(qkv, seq - 1, rope, k1, v1, seq, Hq, D ** -0.5, n, rot)
    a, h = ops.ext().llmint8_attn_up(qkv, seq - 1, rope, k2, v2, seq, Hq, D ** -0.5, n, rot, y, *up.pair_args(), N, up._ACT[act])
    assert torch.equal(k1, k2) and torch.equal(v1, v2)
    assert ((a.view(1, Hq, D).float() - ref.float()).abs() <= 2 ** -7 * ref.float().abs() + 1e-5).all()
    assert torch.equal(h, up.gelu_fused(y, act))


@pytest.mark.parametrize("K", [64, 2048, 2560, 4096])
def test_llmint8_norm_of_both_branches(cuda, K):
    from edgellm import ops
    from edgellm.models.layers import PendingLN
    g = torch.Generator().manual_seed(K)
    x, x2, res = (_rows(g, 1, K, dtype=torch.bfloat16) for _ in range(3))
    g1, b1, g2, b2 = (_rows(g, K, dtype=torch.bfloat16) for _ in range(4))
    m = _l8(g, 272, K)
    h, y = torch.empty_like(x), torch.empty_like(x)
    out = m(PendingLN(x, res, g1, b1, 1e-5, h, y, x2=x2, y_weight=g2, y_bias=b2))
    n1, r = ops.layer_norm(x + x2, g1, b1, 1e-5, res)
    n2, _ = ops.layer_norm(r, g2, b2, 1e-5, None)
    assert torch.equal(h, r) and torch.equal(y, n2) and torch.equal(out, m(n1))


@pytest.mark.parametrize("family", ["gpt_neox", "phi"])                  # two norms of the same row; one
def test_llmint8_decode_steps_agree_with_the_separate_launches(cuda, family, monkeypatch):
    """The layer's wiring around the int8 launches: branches into the next norm and the final norm, the second norm's weights, caches."""
    from edgellm.models import build_model, tiny
    from edgellm.models.decoder import DecoderLayer
    from edgellm.quant import quantize_model
    cfg = tiny(family, num_layers=3, hidden_size=256, num_heads=4, num_kv_heads=4, intermediate_size=4160, rotary_dim=32)
    model, g = build_model(cfg, dtype=torch.bfloat16, device="cuda", seed=3), torch.Generator().manual_seed(4)
    norms = [n for layer in model.layers for n in (layer.norm1, layer.norm2) if n is not None] + [model.final_norm]
    for n in norms:                                                      # (weights of one would hide a norm in another's place)
        n.weight.data.copy_(0.5 + torch.rand(256, generator=g))
        n.bias.data.copy_(0.5 * torch.randn(256, generator=g))
    model, used = quantize_model(model, "llm_int8"), []
    real = DecoderLayer._pair
    monkeypatch.setattr(DecoderLayer, "_pair", lambda self, *a: used.append(self.idx) or real(self, *a))
    one, k1, v1 = _stepped(model, caches=True)
    assert used == [0, 1, 2] * 2
    monkeypatch.setattr(DecoderLayer, "_pair_ok", lambda self, *a: False)
    two, k2, v2 = _stepped(model, caches=True)
    assert used == [0, 1, 2] * 2
    # only the attention's last bf16 rounding differs (2^-9 of a number).  o quantises those rows in steps of some 3 sigma / 127 = 0.024
    # sigma, so about 2^-9 / 0.024 = 8 % of the numbers may move by a step: sqrt(0.08) 0.024 = 0.7 % of a branch a layer, three layers
    for a, b in ((one, two), (k1, k2), (v1, v2)):
        assert (a.float() - b.float()).norm() <= 0.03 * b.float().norm()
    assert two.std() > 0 and torch.isfinite(two).all()
