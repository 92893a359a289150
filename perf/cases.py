"""The work this framework is measured on, as its users have it do.

Two kinds of cases, one per engine:

  "generate"  a dense decoder answers a batch of prompts: ``Generator.generate`` (prefill, then graph-replayed
              decoding with the reference's sampling), at the models, precisions and batch sizes of
              ``bench.py`` and of the reference's own runs;
  "trace"     a layer-spec decoder replays a trace of ragged steps (prompt portions beside decode tokens) through
              ``RaggedEngine.step``, as ``bin/trace_run`` and the continuous-batching scheduler drive it, at the
              sizes of ``bench.py --hybrid-compare``.

Weights are random, made from the seed, but for two things that a trained model has too and that let the whole of a
run be compared: a generating model's output projection is laid out so that each token has one clearly likely
successor, so that the sampled tokens do not hang on the last bit of a logit; and a router's scores follow the token
(a few coordinates of the stream carry a code that the embedding writes, the routers read and no sublayer changes), so
that no choice of experts hangs on the last bit of a score.
"""
import math
import zlib

import torch

import edgellm  # noqa: F401
from edgellm.engine import Generator, SamplingParams
from edgellm.engine.ragged import RaggedEngine
from edgellm.engine.ragged_bench import (NUMIZEN_SIZES, PAGONEX_SIZES, SIZES, VETEVIK_SIZES, hybrid_config, numizen_config,
                                         pagonex_config, vetevik_config)
from edgellm.models import build_model, get_config
from edgellm.models.hybrid import CONVERTERS, build_hybrid, load_into_hybrid
from edgellm.quant import quantize_model, synthetic_calibration

DEV = "cuda:0"
F64 = torch.float64
PAGE = 64


# --------------------------------------------------------------------------- the cases
def _gen(name, model, layers, mode, batch, prompt, new, ragged=False):
    c = dict(kind="generate", model=model, layers=layers, mode=mode, batch=batch, prompt=prompt, new=new, ragged=ragged)
    return dict(c, name=name) if name else c


def _trace(name, family, size, dtype, requests, prompt, portion, new, stagger=0, ragged=False, score=1):
    """``score``: the prompt's last tokens whose logits are wanted (1: the one that chooses the first new token)."""
    c = dict(kind="trace", family=family, size=size, dtype=dtype, requests=requests, prompt=prompt, portion=portion, new=new,
             stagger=stagger, ragged=ragged, score=score)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one question at a time, as the reference evaluates its models: a short prompt, an answer token by token
        _gen("answer llama-3.2-1b bf16", "llama-3.2-1b", 16, "bf16", 1, 32, 64),
        _gen("answer pythia-1b fp16", "pythia-1b", 16, "fp16", 1, 21, 48),
        # the reference's quantised agents: LLM.int8 at batch 1
        _gen("answer phi-2 llm.int8", "phi-2", 32, "llm_int8", 1, 45, 32),
        # bench.py's latency point: Llama-2-7B, SmoothQuant W8A8, one sequence
        _gen("latency llama-2-7b w8a8", "llama-2-7b", 32, "w8a8_smoothquant", 1, 128, 32),
        # bench.py's micro-batch of 256 sequences through one stage of the four-way split
        _gen("batch 256 llama-2-7b w8a8", "llama-2-7b", 8, "w8a8_smoothquant", 256, 128, 32),
        # unequal prompts answered together in bf16 (the four-way bf16 pipeline's stage)
        _gen("ragged 23 llama-2-7b bf16", "llama-2-7b", 8, "bf16", 23, 101, 40, True),
        # a long document before a short answer: one stage of the eight-way Llama-3-8B split
        _gen("document llama-3-8b w8a8", "llama-3-8b", 4, "w8a8_smoothquant", 1, 7967, 8),
        # layer-spec models: one long prompt in one piece, its last part (an answer that is judged) scored token by token
        # (latent attention + delta rule + experts)
        _trace("prompt pagonex w1024", "pagonex", "w1024", "bf16", 1, 4096, 4096, 1, score=100),
        # the longest prompt, at the larger size (full latent attention + gated linear attention + grouped experts)
        _trace("long prompt numizen w2048", "numizen", "w2048", "bf16", 1, 7680, 7680, 1, score=64),
        # serving: unequal prompts arrive one after another, in portions beside the others' decode tokens
        _trace("serving vetevik w2048", "vetevik", "w2048", "bf16", 6, 1100, 512, 24, 2, True),
        # decoding: four sequences token by token after short prompts
        _trace("decode pagonex w1024", "pagonex", "w1024", "bf16", 4, 33, 64, 64),
        # the fp32 kernels: two odd prompts and a short answer (attention beside a state-space mixer)
        _trace("fp32 nudadra w1024", "nudadra", "w1024", "fp32", 2, 777, 512, 16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["answer", "batch", "document", "prompt", "serving", "decode"])
    if kind == "answer":
        model, layers = rng.choice([("llama-3.2-1b", 16), ("pythia-1b", 16), ("phi-2", 32)])
        mode = rng.choice(["bf16", "llm_int8", "w8a8_smoothquant"] if model == "llama-3.2-1b" else ["fp16", "llm_int8", "w8a8_smoothquant"])
        return _gen(None, model, layers, mode, 1, _log(rng, 12, 200), rng.randint(16, 64))
    if kind == "batch":
        mode = rng.choice(["bf16", "w8a8_smoothquant"])
        return _gen(None, "llama-2-7b", rng.choice([4, 8]), mode, _log(rng, 2, 256), _log(rng, 40, 128), rng.randint(16, 32),
                    rng.random() < 0.5)
    if kind == "document":
        return _gen(None, "llama-3-8b", 4, rng.choice(["bf16", "w8a8_smoothquant"]), 1, _log(rng, 500, 7900), rng.randint(2, 8))
    family = rng.choice(["nudadra", "pagonex", "vetevik", "numizen"])
    size = rng.choice(["w1024", "w2048"])
    dtype = "fp32" if size == "w1024" and rng.random() < 0.25 else "bf16"
    if kind == "prompt":
        n = _log(rng, 100, 2000 if dtype == "fp32" else 7600)
        return _trace(None, family, size, dtype, 1, n, n, 1, score=rng.randint(16, 100))
    if kind == "serving":
        return _trace(None, family, size, dtype, rng.randint(2, 6), _log(rng, 100, 1100), rng.choice([128, 256, 512]),
                      rng.randint(8, 24), rng.randint(0, 3), True)
    return _trace(None, family, size, dtype, _log(rng, 1, 16), _log(rng, 8, 128), 512, rng.randint(16, 64))


# --------------------------------------------------------------------------- random numbers by name
def _generator(seed, name):
    return torch.Generator(device=DEV).manual_seed((seed * 1000003 + zlib.crc32(name.encode())) % (2 ** 62))


def _randn(seed, name, *shape):
    return torch.randn(shape, generator=_generator(seed, name), device=DEV, dtype=torch.float32)


def _rand(seed, name, *shape):
    return torch.rand(shape, generator=_generator(seed, name), device=DEV, dtype=torch.float32)


def _ints(seed, name, high, n):
    g = torch.Generator().manual_seed((seed * 1000003 + zlib.crc32(name.encode())) % (2 ** 62))
    return torch.randint(0, high, (n,), generator=g).tolist()


def _lengths(case, n):
    """Prompt lengths of the ``n`` sequences: equal, or spread below the longest."""
    P = case["prompt"]
    if not case["ragged"]:
        return [P] * n
    if case["kind"] == "generate":                     # an answer is longer than the prompts' lengths differ
        spread = max(1, min(P - 1, case["new"] - 1))
    else:
        spread = max(1, P // 2)
    return [P - (r * 37) % spread for r in range(n)]


# --------------------------------------------------------------------------- dense decoders
def _dense_config(case):
    cfg = get_config(case["model"]).replace(num_layers=case["layers"])
    need = case["prompt"] + case["new"]
    return cfg if need <= cfg.max_position_embeddings else cfg.replace(max_position_embeddings=need)


def _dense_tensor(cfg, seed, name, shape):
    """One parameter in fp32.  Embedding rows are as large as the stream that the sublayers add to; projections keep
    their input's size; each sublayer adds about as much as half the embedding's size over the whole depth."""
    if name.endswith("norm1.weight") or name.endswith("norm2.weight"):
        return 1.0 + 0.1 * _randn(seed, name, *shape)
    if name == "final_norm.weight":
        w = 1.0 + 0.05 * _randn(seed, name, *shape)
        return w * _sign(cfg, seed) if cfg.tie_word_embeddings else w
    if name.endswith("bias"):
        return 0.05 * _randn(seed, name, *shape)
    if name == "embed":
        e = _randn(seed, name, *shape)
        if cfg.tie_word_embeddings:                    # neighbours 2m, 2m + 1 follow one another
            e[1::2] = e[0::2] * _sign(cfg, seed)
        return e
    if name == "lm_head.weight":                       # row j: the token whose successor is j
        e = _dense_tensor(cfg, seed, "embed", shape).to(torch.bfloat16).float()
        return e[(torch.arange(shape[0], device=DEV) - _step(cfg)) % shape[0]] * shape[1] ** -0.5
    w = _randn(seed, name, *shape) * shape[1] ** -0.5
    return w * (1.5 * cfg.num_layers ** -0.5) if name.endswith("o.weight") or name.endswith("down.weight") else w


def _sign(cfg, seed):
    return torch.where(_rand(seed, "sign", cfg.hidden_size) < 0.5, -1.0, 1.0)


def _step(cfg):
    return 7919                                        # odd and prime: a chain through the whole vocabulary


def _successor(cfg, t):
    return t ^ 1 if cfg.tie_word_embeddings else (t + _step(cfg)) % cfg.vocab_size


def _dense_shapes(cfg):
    W, F = cfg.hidden_size, cfg.intermediate_size
    s = {"embed": (cfg.vocab_size, W), "final_norm.weight": (W,)}
    ln = cfg.norm == "layer"
    if ln:
        s["final_norm.bias"] = (W,)
    if not cfg.tie_word_embeddings:
        s["lm_head.weight"] = (cfg.vocab_size, W)
    if cfg.lm_head_bias:
        s["lm_head.bias"] = (cfg.vocab_size,)
    for i in range(cfg.num_layers):
        p = "layers.%d." % i
        for n in ("norm1",) if cfg.shared_input_norm else ("norm1", "norm2"):
            s[p + n + ".weight"] = (W,)
            if ln:
                s[p + n + ".bias"] = (W,)
        up = 2 * F if cfg.act == "silu_glu" else F
        for n, rows, cols, bias in (("attn.qkv", cfg.qkv_size, W, cfg.qkv_bias), ("attn.o", W, cfg.q_size, cfg.o_bias),
                                    ("mlp.up", up, W, cfg.mlp_bias), ("mlp.down", W, F, cfg.mlp_bias)):
            s[p + n + ".weight"] = (rows, cols)
            if bias:
                s[p + n + ".bias"] = (rows,)
    return s


def _dense_dtype(case):
    return torch.float16 if case["mode"] == "fp16" else torch.bfloat16


def _dense_prompts(case, cfg, seed):
    return [_ints(seed, "prompt%d" % b, cfg.vocab_size, n) for b, n in enumerate(_lengths(case, case["batch"]))]


def _prepare_dense(case, seed):
    cfg = _dense_config(case)
    model = build_model(cfg, dtype=_dense_dtype(case), device=DEV, seed=None)
    params = dict(model.named_parameters())
    for name, shape in _dense_shapes(cfg).items():
        params[name].data.copy_(_dense_tensor(cfg, seed, name, shape))
    del params
    if case["mode"] not in ("bf16", "fp16"):
        calib = synthetic_calibration(cfg, n=2, T=64, device=DEV, seed=seed) if case["mode"] == "w8a8_smoothquant" else None
        model = quantize_model(model, case["mode"], calib)
    gen = Generator(model, max_batch=case["batch"], max_seq=case["prompt"] + case["new"])
    sp = SamplingParams(max_new_tokens=case["new"], temperature=0.7, top_k=50, top_p=0.9, repetition_penalty=1.1)
    return dict(kind="generate", gen=gen, sampling=sp, prompts=_dense_prompts(case, cfg, seed), seed=seed & 0xFFFF)


def _run_dense(s):
    gen = s["gen"]
    res = gen.generate(s["prompts"], s["sampling"], seed=s["seed"])
    return {"tokens": torch.tensor(res.tokens), "logits": gen._run["prefill_logits"], "k": gen.kv.k, "v": gen.kv.v}


def _silu(z):
    return z * torch.sigmoid(z)


def _frequencies(dims, base, scaling):
    """(angle per position of each pair, gain of cos and sin)."""
    f = base ** (-torch.arange(0, dims, 2, dtype=F64, device=DEV) / dims)
    kind = (scaling or {}).get("rope_type")
    if kind == "llama3":
        old, wave = scaling["original_max_position_embeddings"], 2 * math.pi / f
        low, high = old / scaling["low_freq_factor"], old / scaling["high_freq_factor"]
        mix = ((old / wave - scaling["low_freq_factor"]) / (scaling["high_freq_factor"] - scaling["low_freq_factor"])).clamp(0, 1)
        part = (1 - mix) * f / scaling["factor"] + mix * f
        return torch.where(wave > low, f / scaling["factor"], torch.where(wave < high, f, part)), 1.0
    if kind == "yarn":
        where = lambda turns: dims * math.log(scaling["original"] / (2 * math.pi * turns)) / (2 * math.log(base))  # noqa: E731
        lo, hi = max(math.floor(where(scaling["fast"])), 0), min(math.ceil(where(scaling["slow"])), dims - 1)
        ramp = ((torch.arange(dims // 2, dtype=F64, device=DEV) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        return f / scaling["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(scaling["factor"]) + 1.0
    return f, 1.0


def _rotate(x, dims, base, scaling=None, neighbours=False):
    """x [T, heads, D] at positions 0..T-1: coordinate pairs (i, i + dims / 2), or (2 i, 2 i + 1)."""
    if not dims:
        return x
    f, gain = _frequencies(dims, base, scaling)
    a = torch.arange(x.shape[0], dtype=F64, device=DEV)[:, None] * f[None]
    c, s = (a.cos() * gain)[:, None], (a.sin() * gain)[:, None]
    y = x.clone()
    if neighbours:
        u, v = x[..., 0:dims:2], x[..., 1:dims:2]
        y[..., 0:dims:2], y[..., 1:dims:2] = u * c - v * s, v * c + u * s
    else:
        u, v = x[..., :dims // 2], x[..., dims // 2:dims]
        y[..., :dims // 2], y[..., dims // 2:dims] = u * c - v * s, v * c + u * s
    return y


def _attention(q, k, v, scale, sees, score=None, sink=None):
    """q [T, H, D], k / v [N, G, D]; ``sees``(query rows, key rows) -> bool; ``score`` changes the scaled scores
    [H, t, N]; exp(sink) joins the denominator."""
    T, H, N = q.shape[0], q.shape[1], k.shape[0]
    kk = k.repeat_interleave(H // k.shape[1], 1).permute(1, 2, 0).contiguous()
    vv = v.repeat_interleave(H // v.shape[1], 1).permute(1, 0, 2).contiguous()
    out, keys = [], torch.arange(N, device=DEV)
    for t0 in range(0, T, 512):
        rows = torch.arange(t0, min(T, t0 + 512), device=DEV)
        s = torch.matmul(q[rows].permute(1, 0, 2).contiguous(), kk) * scale
        if score is not None:
            s = score(s, rows, keys)
        s = s.masked_fill(~sees(rows[:, None], keys[None, :])[None], -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[:, None, None].expand(-1, len(rows), 1)], -1)
        p = torch.softmax(s, -1)[..., :N]
        out.append(torch.matmul(p, vv).permute(1, 0, 2))
    return torch.cat(out, 0)


def _causal(i, j):
    return j <= i


def _layer_norm(x, w, b, eps):
    x = x - x.mean(-1, keepdim=True)
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w + b


def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _gelu(z, tanh):
    return torch.nn.functional.gelu(z, approximate="tanh" if tanh else "none")


def _exact_dense(case, seed):
    cfg = _dense_config(case)
    dt = _dense_dtype(case)
    shapes = _dense_shapes(cfg)
    get = lambda n: _dense_tensor(cfg, seed, n, shapes[n]).to(dt).to(F64) if n in shapes else None  # noqa: E731
    prompts, new = _dense_prompts(case, cfg, seed), case["new"]
    chains = []
    for p in prompts:
        seq = list(p)
        while len(seq) < len(p) + new - 1:
            seq.append(_successor(cfg, seq[-1]))
        chains.append(seq)
    B, S, D, G, H = len(prompts), case["prompt"] + new, cfg.head_dim, cfg.num_kv_heads, cfg.num_heads
    norm = lambda x, n: (_rms(x, cfg.norm_eps) * get(n + ".weight") if cfg.norm == "rms" else  # noqa: E731
                         _layer_norm(x, get(n + ".weight"), get(n + ".bias"), cfg.norm_eps))
    lens = [len(c) for c in chains]
    ids = torch.tensor([t for c in chains for t in c], device=DEV)
    x = get("embed")[ids]
    kc, vc = (torch.zeros(cfg.num_layers, B, G, S, D, dtype=F64, device=DEV) for _ in range(2))

    def project(h, w, b, rows=16384):
        y = torch.cat([h[r:r + rows] @ w.T for r in range(0, h.shape[0], rows)])
        return y if b is None else y + b

    def feed_forward(h, p):
        wu, bu, wd, bd = (get(p + n) for n in ("mlp.up.weight", "mlp.up.bias", "mlp.down.weight", "mlp.down.bias"))
        out = []
        for r in range(0, h.shape[0], 8192):
            u = project(h[r:r + 8192], wu, bu)
            if cfg.act == "silu_glu":
                g, u = u.chunk(2, -1)
                u = _silu(g) * u
            else:
                u = _gelu(u, cfg.act == "gelu_tanh")
            out.append(project(u, wd, bd))
        return torch.cat(out)

    def attend(h, p, i):
        qkv = project(h, get(p + "attn.qkv.weight"), get(p + "attn.qkv.bias"))
        out, at = [], 0
        for b, n in enumerate(lens):
            q, k, v = torch.split(qkv[at:at + n], [H * D, G * D, G * D], -1)
            q = _rotate(q.reshape(n, H, D), cfg.rotary_dim, cfg.rope_theta, cfg.rope_scaling)
            k = _rotate(k.reshape(n, G, D), cfg.rotary_dim, cfg.rope_theta, cfg.rope_scaling)
            v = v.reshape(n, G, D)
            kc[i, b, :, :n], vc[i, b, :, :n] = k.permute(1, 0, 2), v.permute(1, 0, 2)
            out.append(_attention(q, k, v, D ** -0.5, _causal).reshape(n, H * D))
            at += n
        return project(torch.cat(out), get(p + "attn.o.weight"), get(p + "attn.o.bias"))

    for i in range(cfg.num_layers):
        p = "layers.%d." % i
        if cfg.parallel_residual:
            h1 = norm(x, p + "norm1")
            h2 = h1 if cfg.shared_input_norm else norm(x, p + "norm2")
            x = x + attend(h1, p, i) + feed_forward(h2, p)
        else:
            x = x + attend(norm(x, p + "norm1"), p, i)
            x = x + feed_forward(norm(x, p + "norm2"), p)
    ends = torch.tensor(lens, device=DEV).cumsum(0)
    rows = torch.stack([ends - new + j for j in range(new)], 1)          # the row that chooses new token j
    h = norm(x, "final_norm")
    head = get("embed" if cfg.tie_word_embeddings else "lm_head.weight")
    bias = get("lm_head.bias")
    tokens = torch.stack([project(h[rows[:, j]], head, bias).argmax(-1) for j in range(new)], 1)
    # SmoothQuant moves scales between the value projection and the one after it: the cached values are its own
    return {"tokens": tokens.cpu(), "logits": project(h[rows[:, 0]], head, bias), "k": kc,
            "v": None if case["mode"] == "w8a8_smoothquant" else vc}


# --------------------------------------------------------------------------- layer-spec decoders
_FAMILIES = {"nudadra": (SIZES, hybrid_config), "pagonex": (PAGONEX_SIZES, pagonex_config),
             "vetevik": (VETEVIK_SIZES, vetevik_config), "numizen": (NUMIZEN_SIZES, numizen_config)}


def _spec_config(case):
    sizes, make = _FAMILIES[case["family"]]
    return make(sizes[case["size"]])


def _expert_shapes(p, m, W, gated):
    names = ("gate", "up") if gated else ("up",)
    s = {p + "router": (m.experts, W)}
    for e in ["e%d" % k for k in range(m.experts)] + (["shared"] if m.shared_ff else []):
        ff = m.shared_ff if e == "shared" else m.ff
        s.update({"%s%s.%s" % (p, e, n): (ff, W) for n in names})
        s["%s%s.down" % (p, e)] = (W, ff)
    return s


def _spec_shapes(family, cfg):
    """Checkpoint tensors of a layer-spec model: name -> shape."""
    W, V = cfg.hidden_size, cfg.vocab_size
    s = {"embed": (V, W)}
    if family != "vetevik":                            # Vetevik's embedding is also its output projection
        s["head"] = (V, W)
    if family == "nudadra":
        s["final.norm"] = ()
    else:
        s["final.norm"] = (W,)
    if family in ("pagonex", "numizen"):
        s["final.norm.b"] = (W,)
    if family == "pagonex":
        s["bigram"] = (cfg.bigram["buckets"] + 1, W)
    if family == "numizen":
        s.update({"pos": (cfg.max_position_embeddings, W), "final.norm.alpha": ()})
    for i, l in enumerate(cfg.layer_specs):
        p = "l%d." % i
        M, F = p + "mix.", p + "mlp."
        if family == "nudadra":
            a, m = l.attn, l.ssd
            L, R = M + "left.", M + "right."
            s.update({p + "norm1": (), L + "q": (a.heads * a.dim, W), L + "k": (a.kv_heads * a.dim, W),
                      L + "v": (a.kv_heads * a.vdim, W), L + "g": (a.heads, W), L + "o": (W, a.heads * a.vdim), L + "out": (W,),
                      R + "in": (m.in_size, W), R + "conv": (m.conv_channels, m.conv), R + "conv.b": (m.conv_channels,),
                      R + "dt_bias": (m.heads,), R + "A_log": (m.heads,), R + "D": (m.heads,), R + "norm": (m.inner,),
                      R + "o": (W, m.inner), R + "out": (W,), F + "up": (l.ff, W), F + "down": (W, l.ff)})
            continue
        if family == "pagonex":
            s.update({p + n: (W,) for n in ("norm1", "norm1.b", "norm2", "norm2.b")})
            s.update({p + n: (W, cfg.canon_taps) for n in ("canon1", "canon2")})
        elif family == "vetevik":
            s.update({p + n: (W,) for n in ("norm1", "norm1b", "norm2", "norm2b")})
        else:
            s.update({p + n: (W,) for n in ("norm1", "norm1.b", "norm2", "norm2.b", "ls1", "ls2")})
            s.update({p + n: () for n in ("norm1.alpha", "norm2.alpha")})
        if l.latent is not None:
            a = l.latent
            s.update({M + "dq": (a.q_rank, W), M + "dq.norm": (a.q_rank,), M + "uq": (a.heads * (a.dim + a.rot_dim), a.q_rank),
                      M + "uk": (a.heads * a.dim, a.kv_rank), M + "uv": (a.heads * a.vdim, a.kv_rank), M + "o": (W, a.heads * a.vdim)})
            if a.kv_from is None:
                s.update({M + "dkv": (a.kv_rank + a.rot_dim, W), M + "dkv.norm": (a.kv_rank,)})
            if a.gate:
                s[M + "g"] = (a.heads * a.vdim, W)
        elif l.delta is not None:
            d = l.delta
            GN, HP = d.kv_heads * d.dim, d.heads * d.vdim
            s.update({M + "q": (GN, W), M + "k": (GN, W), M + "v": (HP, W), M + "b": (d.heads, W), M + "q.conv": (GN, d.conv),
                      M + "k.conv": (GN, d.conv), M + "v.conv": (HP, d.conv), M + "A_log": (d.heads,), M + "norm": (d.vdim,),
                      M + "o": (W, HP)})
            if d.decay == "head":
                s.update({M + "a": (d.heads, W), M + "g": (HP, W), M + "dt_bias": (d.heads,)})
            else:
                s.update({M + "a1": (d.decay_rank, W), M + "a2": (d.heads * d.dim, d.decay_rank), M + "g1": (d.gate_rank, W),
                          M + "g2": (HP, d.gate_rank), M + "dt_bias": (d.heads * d.dim,)})
        elif l.chunk_attn is not None:
            a = l.chunk_attn
            s.update({M + "q": (a.heads * a.dim, W), M + "k": (a.kv_heads * a.dim, W), M + "g": (a.heads * a.dim, W),
                      M + "sink": (a.heads,), M + "o": (W, a.heads * a.dim)})
        else:
            g = l.gla
            s.update({M + n: (g.heads * g.dim, W) for n in ("q", "k")})
            s.update({M + n: (g.heads * g.vdim, W) for n in ("v", "g")})
            s.update({M + "a1": (g.decay_rank, W), M + "a2": (g.heads * g.dim, g.decay_rank), M + "a2.b": (g.heads * g.dim,),
                      M + "norm": (g.vdim,), M + "o": (W, g.heads * g.vdim)})
        if l.moe is not None:
            s.update(_expert_shapes(F, l.moe, W, family != "numizen"))
            if family == "numizen":
                s.update({F + "correction": (l.moe.experts,), F + "shared.sg": (1, W)})
        elif l.ff:
            s.update({F + "gate": (l.ff, W), F + "up": (l.ff, W), F + "down": (W, l.ff)})
    return s


def _codes(cfg):
    """How many coordinates of the stream carry the routers' code: one per expert."""
    return max((l.moe.experts for l in cfg.layer_specs if l.moe is not None), default=0)


def _spec_tensor(cfg, seed, name, shape):
    family, C = cfg.arch, _codes(cfg)
    leaf = name.split(".")[-1]
    if name.endswith("router"):                        # expert e reads one code coordinate, another one in every layer
        v = torch.zeros(shape, device=DEV)
        e = torch.arange(shape[0], device=DEV)
        v[e, (e + 5 * int(name[1:name.index(".")])) % C] = 6.0 if family == "numizen" else 2.0
        return v.to(torch.bfloat16)
    r = _randn(seed, name, *shape)
    if name == "embed":
        v = r
    elif name == "bigram":
        v = 0.5 * r
    elif name == "pos":
        v = 0.3 * r
    elif leaf == "A_log":
        v = torch.log(1.0 + 7.0 * _rand(seed, name, *shape))
    elif leaf == "dt_bias":
        v = torch.log(torch.expm1(0.01 + 0.2 * _rand(seed, name, *shape)))
    elif leaf == "alpha":
        v = 0.5 + 0.1 * r
    elif leaf in ("ls1", "ls2"):
        v = 0.5 + 0.1 * r
    elif name.endswith("a2.b"):                        # decays that keep a token for tens to hundreds of steps
        v = 2.0 + r
    elif leaf == "correction":
        v = 1e-4 * r
    elif leaf == "sink":
        v = r
    elif leaf in ("canon1", "canon2"):
        v = 0.3 * r
    elif leaf == "b" and len(shape) == 1:
        v = 0.1 * r
    elif leaf in ("norm1b", "norm2b") or (family == "pagonex" and leaf in ("norm1", "norm2")):
        v = 0.5 + 0.05 * r                             # norms of sublayers' outputs: a part of the stream's own size
    elif leaf in ("norm", "norm1", "norm2", "out", "D"):
        v = 1.0 + 0.1 * r
    else:                                              # projections and convolutions
        v = r * shape[-1] ** -0.5
    if C and name == "embed":                          # each token's code: evenly spaced levels in an order of its own
        levels = torch.linspace(-1.7, 1.7, C, device=DEV)
        v[:, :C] = levels[_rand(seed, "code", shape[0], C).argsort(-1)]
    elif C and (name in ("bigram", "pos") or leaf in ("canon1", "canon2", "ls1", "ls2", "norm1b", "norm2b")
                or (family == "pagonex" and name[0] == "l" and ".norm" in name)):
        v[(slice(None), slice(C)) if name in ("bigram", "pos") else slice(C)] = 0.0   # what adds to the stream leaves the code alone
    elif C and name[0] == "l" and ".norm2" in name and not name.endswith("alpha"):
        v[:C] = 0.0 if leaf == "b" else 1.0            # what the router reads keeps the code's order
    return v.to(torch.bfloat16)


def _spec_tensors(case, seed):
    cfg = _spec_config(case)
    return cfg, {n: _spec_tensor(cfg, seed, n, s) for n, s in _spec_shapes(case["family"], cfg).items()}


def _spec_tokens(case, cfg, seed):
    """Per request (prompt, the tokens that its decode steps bring)."""
    R = case["requests"]
    return [(_ints(seed, "prompt%d" % r, cfg.vocab_size, n), _ints(seed, "answer%d" % r, cfg.vocab_size, case["new"] - 1))
            for r, n in enumerate(_lengths(case, R))]


def _schedule(case):
    """Steps of (request, first position, tokens, which of them want logits): a request starts ``stagger`` steps after
    the one before."""
    lens, left = _lengths(case, case["requests"]), []
    done = [0] * len(lens)
    step = 0
    while any(d < n + case["new"] - 1 for d, n in zip(done, lens)):
        now = []
        for r, n in enumerate(lens):
            if step < r * case["stagger"] or done[r] >= n + case["new"] - 1:
                continue
            take = min(case["portion"], n - done[r]) if done[r] < n else 1
            first = n - min(case["score"], n)          # every token from here on wants its logits
            now.append((r, done[r], take, list(range(max(0, first - done[r]), take))))
            done[r] += take
        left.append(now)
        step += 1
    return left


def _spec_dtype(case):
    return torch.float32 if case["dtype"] == "fp32" else torch.bfloat16


def _state_runs(cfg):
    """The layers that carry a recurrent state."""
    return [i for i, l in enumerate(cfg.layer_specs) if l.ssd is not None or l.delta is not None or l.gla is not None]


def _prepare_spec(case, seed):
    cfg, tensors = _spec_tensors(case, seed)
    model = build_hybrid(cfg, _spec_dtype(case), DEV, seed=None)
    load_into_hybrid(model, CONVERTERS[case["family"]][0](cfg, tensors))
    del tensors
    sizes = _lengths(case, case["requests"])
    tokens = sum((n + case["new"] + PAGE - 1) // PAGE * PAGE for n in sizes)
    eng = RaggedEngine(model, tokens, slots=case["requests"], page=PAGE)
    full = [p + a for p, a in _spec_tokens(case, cfg, seed)]
    steps = [[(r, full[r][at:at + n], want) for r, at, n, want in now] for now in _schedule(case)]
    return dict(kind="trace", engine=eng, steps=steps, requests=case["requests"], state_runs=_state_runs(cfg))


def _run_spec(s):
    eng = s["engine"]
    logits = [eng.step(entries) for entries in s["steps"]]
    slots = [eng.live[r] for r in range(s["requests"])]
    states = [eng.cache.run(i).ssm[slots] for i in s["state_runs"]]
    for r in range(s["requests"]):
        eng.close(r)
    return {"logits": torch.cat(logits), "states": states}


def _conv(x, w):
    """Causal depthwise convolution over time; the last tap meets the current token."""
    taps = w.shape[1]
    pad = torch.cat([x.new_zeros(taps - 1, x.shape[1]), x])
    return sum(pad[j:j + x.shape[0]] * w[:, j] for j in range(taps))


def _scan(q, k, v, decay, beta=None):
    """S <- decay S + k u^T with u = v, or beta (v - S^T k) of the decayed S; o = S^T q.  q / k [T, H, N], v [T, H, P],
    decay [T, H, N or 1], beta [T, H] -> (o [T, H, P], S [H, N, P])."""
    T, H, N = k.shape
    S = torch.zeros(H, N, v.shape[2], dtype=F64, device=DEV)
    out = torch.empty_like(v)
    decay, kc = decay[..., None], k[..., None].contiguous()
    qr, kr = q[:, :, None, :].contiguous(), k[:, :, None, :].contiguous()
    for t in range(T):
        S = S * decay[t]
        u = v[t][:, None]
        if beta is not None:
            u = (u - torch.matmul(kr[t], S)) * beta[t][:, None, None]
        S = torch.baddbmm(S, kc[t], u)
        out[t] = torch.matmul(qr[t], S)[:, 0]
    return out, S


def _softplus(z):
    return torch.nn.functional.softplus(z, threshold=1e9)


def _experts(h, idx, wts, act, on_input=False):
    """sum over the chosen experts: ``act``(rows, expert) is one expert's output."""
    out = torch.zeros_like(h)
    for e in idx.unique().tolist():
        t, c = (idx == e).nonzero(as_tuple=True)
        w = wts[t, c][:, None]
        out.index_add_(0, t, act(h[t] * w, e) if on_input else act(h[t], e) * w)
    return out


def _latent_attention(h, w, M, a, eps, kept):
    T = h.shape[0]
    q = ((_rms(h @ w[M + "dq"].T, eps) * w[M + "dq.norm"]) @ w[M + "uq"].T).reshape(T, a.heads, a.dim + a.rot_dim)
    turn = lambda x: _rotate(x, a.rot_dims, a.rot_base, a.rot_scaling, neighbours=True)  # noqa: E731
    if a.kv_from is None:
        d = h @ w[M + "dkv"].T
        kept = _rms(d[:, :a.kv_rank], eps) * w[M + "dkv.norm"], turn(d[:, None, a.kv_rank:])
    c, shared = kept
    k = torch.cat([(c @ w[M + "uk"].T).reshape(T, a.heads, a.dim), shared.expand(-1, a.heads, -1)], -1)
    v = (c @ w[M + "uv"].T).reshape(T, a.heads, a.vdim)
    q = torch.cat([q[..., :a.dim], turn(q[..., a.dim:])], -1)
    sees = _causal if a.window is None else lambda i, j: (j <= i) & (i - j < a.window)
    o = _attention(q, k, v, a.scale, sees).reshape(T, -1)
    if a.gate:
        o = o * torch.sigmoid(h @ w[M + "g"].T)
    return o @ w[M + "o"].T, kept


def _delta_mixer(h, w, M, d, eps):
    T, G, H, N, P = h.shape[0], d.kv_heads, d.heads, d.dim, d.vdim
    short = lambda n: _silu(_conv(h @ w[M + n].T, w[M + n + ".conv"]))  # noqa: E731
    unit = lambda x: x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    spread = lambda x: x.repeat_interleave(H // G, 1)  # noqa: E731
    q, k = spread(unit(short("q").reshape(T, G, N)) * N ** -0.5), spread(unit(short("k").reshape(T, G, N)))
    v, beta = short("v").reshape(T, H, P), torch.sigmoid(h @ w[M + "b"].T)
    rate = torch.exp(w[M + "A_log"])
    if d.decay == "head":
        g = torch.exp(-rate * _softplus(h @ w[M + "a"].T + w[M + "dt_bias"]))[..., None]
        gate = _silu(h @ w[M + "g"].T)
    else:
        z = (h @ w[M + "a1"].T) @ w[M + "a2"].T + w[M + "dt_bias"]
        g = torch.exp(-rate[:, None] * _softplus(z).reshape(T, H, N))
        gate = torch.sigmoid((h @ w[M + "g1"].T) @ w[M + "g2"].T)
    o, S = _scan(q, k, v, g, beta)
    return ((_rms(o, eps) * w[M + "norm"]).reshape(T, -1) * gate) @ w[M + "o"].T, S


def _forward_nudadra(cfg, w, ids):
    eps, x, states = cfg.norm_eps, w["embed"][ids] * cfg.embed_scale, []
    T = len(ids)
    for i, l in enumerate(cfg.layer_specs):
        p = "l%d." % i
        h = _rms(x, eps) * w[p + "norm1"]
        a, m, L, R = l.attn, l.ssd, p + "mix.left.", p + "mix.right."
        turn = lambda y: _rotate(y, a.rot_dims, a.rot_base, a.rot_scaling)  # noqa: E731
        q, k = turn((h @ w[L + "q"].T).reshape(T, a.heads, -1)), turn((h @ w[L + "k"].T).reshape(T, a.kv_heads, -1))
        v = (h @ w[L + "v"].T).reshape(T, a.kv_heads, -1)
        n = T // a.pool                                # keys: the tokens, then the blocks' means
        blocks = lambda y: torch.cat([y, y[:n * a.pool].reshape(n, a.pool, *y.shape[1:]).mean(1)])  # noqa: E731

        def sees(i_, j):
            token = (j < T) & (j <= i_) & (i_ - j < a.window)
            return token | ((j >= T) & ((j - T) * a.pool + a.pool - 1 <= i_ - a.window))
        o = _attention(q, blocks(k), blocks(v), a.scale, sees) * torch.sigmoid(h @ w[L + "g"].T)[..., None]
        left = o.reshape(T, -1) @ w[L + "o"].T
        u = h @ w[R + "in"].T
        z, xbc, dt = torch.split(u, [m.inner, m.conv_channels, m.heads], -1)
        xbc = _silu(_conv(xbc, w[R + "conv"]) + w[R + "conv.b"])
        xs, Bm, Cm = torch.split(xbc, [m.inner, m.groups * m.state, m.groups * m.state], -1)
        xs = xs.reshape(T, m.heads, m.vdim)
        spread = lambda y: y.reshape(T, m.groups, m.state).repeat_interleave(m.heads // m.groups, 1)  # noqa: E731
        dt = _softplus(dt + w[R + "dt_bias"])
        y, S = _scan(spread(Cm), spread(Bm), xs * dt[..., None], torch.exp(-torch.exp(w[R + "A_log"]) * dt)[..., None])
        y = (y + w[R + "D"][:, None] * xs).reshape(T, -1) * _silu(z)
        y = _rms(y.reshape(T, m.norm_groups, -1), eps).reshape(T, -1) * w[R + "norm"]
        right = y @ w[R + "o"].T
        f = torch.relu(h @ w[p + "mlp.up"].T) ** 2 @ w[p + "mlp.down"].T
        x = x + 0.5 * (_rms(left, eps) * w[L + "out"] + _rms(right, eps) * w[R + "out"]) + f
        states.append(S)
    return _rms(x, eps) * w["final.norm"], states


def _forward_pagonex(cfg, w, ids):
    eps, big, kept, states = cfg.norm_eps, cfg.bigram, {}, []
    prev = torch.cat([ids[:1], ids[:-1]])
    pair = (prev * big["mul_prev"] + ids * big["mul_cur"]) % big["buckets"]
    pair[0] = big["buckets"]
    x = w["embed"][ids] + w["bigram"][pair]
    for i, l in enumerate(cfg.layer_specs):
        p, m = "l%d." % i, l.moe
        h = x + _conv(x, w[p + "canon1"])
        if l.latent is not None:
            y, kept[i] = _latent_attention(h, w, p + "mix.", l.latent, eps, kept.get(l.latent.kv_from))
        else:
            y, S = _delta_mixer(h, w, p + "mix.", l.delta, eps)
            states.append(S)
        x = x + _layer_norm(y, w[p + "norm1"], w[p + "norm1.b"], eps)
        h = x + _conv(x, w[p + "canon2"])

        def unit(z, name, limit):
            g = (z @ w[name + ".gate"].T).clamp(max=limit)
            u = (z @ w[name + ".up"].T).clamp(-limit, limit)
            return (g * torch.sigmoid(1.702 * g) * (u + 1)) @ w[name + ".down"].T
        s, idx = torch.softmax(h @ w[p + "mlp.router"].T, -1).topk(m.top, -1)
        y = _experts(h, idx, s / (s.sum(-1, keepdim=True) + 1e-20) * m.scale, lambda z, e: unit(z, "%smlp.e%d" % (p, e), m.limit))
        y = y + unit(h, p + "mlp.shared", m.shared_limit)
        x = x + _layer_norm(y, w[p + "norm2"], w[p + "norm2.b"], eps)
    return _layer_norm(x, w["final.norm"], w["final.norm.b"], eps), states


def _forward_vetevik(cfg, w, ids):
    eps, states, x = cfg.norm_eps, [], w["embed"][ids]
    T = len(ids)
    norm = lambda y, n: _rms(y.reshape(T, cfg.norm_groups, -1), eps).reshape(T, -1) * w[n]  # noqa: E731
    for i, l in enumerate(cfg.layer_specs):
        p, m = "l%d." % i, l.moe
        h = norm(x, p + "norm1")
        if l.chunk_attn is not None:
            a, M = l.chunk_attn, p + "mix."
            q, k = (h @ w[M + "q"].T).reshape(T, a.heads, -1), (h @ w[M + "k"].T).reshape(T, a.kv_heads, -1)
            slope = 2.0 ** (-8.0 * torch.arange(1, a.heads + 1, dtype=F64, device=DEV) / a.heads)
            score = lambda s, i_, j: (a.softcap * torch.tanh(s / a.softcap)  # noqa: E731
                                      - slope[:, None, None] * (i_[:, None] - j[None, :]).to(F64))
            sees = lambda i_, j: (j <= i_) & (j // a.chunk == i_ // a.chunk)  # noqa: E731
            o = _attention(q, k, k, a.scale, sees, score, w[M + "sink"]).reshape(T, -1)
            y = (o * torch.sigmoid(h @ w[M + "g"].T)) @ w[M + "o"].T
        else:
            y, S = _delta_mixer(h, w, p + "mix.", l.delta, eps)
            states.append(S)
        x = x + cfg.residual_mult * norm(y, p + "norm1b")
        h = norm(x, p + "norm2")
        s, idx = torch.sigmoid(h @ w[p + "mlp.router"].T).topk(m.top, -1)

        def unit(z, e):
            n = "%smlp.e%d" % (p, e)
            return (_silu(z @ w[n + ".gate"].T) * (z @ w[n + ".up"].T)) @ w[n + ".down"].T
        x = x + cfg.residual_mult * norm(_experts(h, idx, s, unit, on_input=True), p + "norm2b")
    return norm(x, "final.norm"), states


def _forward_numizen(cfg, w, ids):
    eps, states, T = cfg.norm_eps, [], len(ids)
    x = w["embed"][ids] + w["pos"][:T]
    norm = lambda y, n: torch.tanh(w[n + ".alpha"] * y) * w[n] + w[n + ".b"]  # noqa: E731
    for i, l in enumerate(cfg.layer_specs):
        p, m = "l%d." % i, l.moe
        M, F = p + "mix.", p + "mlp."
        h = norm(x, p + "norm1")
        if l.latent is not None:
            y, _ = _latent_attention(h, w, M, l.latent, eps, None)
        else:
            g = l.gla
            q, k, v = ((h @ w[M + n].T).reshape(T, g.heads, -1) for n in ("q", "k", "v"))
            a = (h @ w[M + "a1"].T) @ w[M + "a2"].T + w[M + "a2.b"]
            decay = torch.exp(-_softplus(-a) / g.tau).reshape(T, g.heads, g.dim)
            o, S = _scan(q * g.dim ** -0.5, k, v, decay)
            y = ((_rms(o, eps) * w[M + "norm"]).reshape(T, -1) * _silu(h @ w[M + "g"].T)) @ w[M + "o"].T
            states.append(S)
        y = y * w[p + "ls1"]
        h = norm(x, p + "norm2")
        if m is None:
            f = (_gelu(h @ w[F + "gate"].T, True) * (h @ w[F + "up"].T)) @ w[F + "down"].T
        else:
            s = torch.softmax(h @ w[F + "router"].T, -1)
            c = s + w[F + "correction"]
            best = c.reshape(T, m.groups, -1).amax(-1).topk(m.groups_keep, -1).indices
            size = m.experts // m.groups
            inside = (torch.arange(m.experts, device=DEV)[None, :, None] // size == best[:, None, :]).any(-1)
            idx = c.masked_fill(~inside, -math.inf).topk(m.top, -1).indices
            wt = s.gather(1, idx)
            unit = lambda z, n: torch.relu(z @ w[n + ".up"].T) ** 2 @ w[n + ".down"].T  # noqa: E731
            f = _experts(h, idx, wt / (wt.sum(-1, keepdim=True) + 1e-20), lambda z, e: unit(z, "%se%d" % (F, e)))
            f = f + unit(h, F + "shared") * torch.sigmoid(h @ w[F + "shared.sg"].T)
        x = x + y + f * w[p + "ls2"]
    return norm(x, "final.norm"), states


_FORWARD = {"nudadra": _forward_nudadra, "pagonex": _forward_pagonex, "vetevik": _forward_vetevik, "numizen": _forward_numizen}


def _exact_spec(case, seed):
    cfg, tensors = _spec_tensors(case, seed)
    w = {n: t.to(F64) for n, t in tensors.items()}
    del tensors
    hidden, states = [], []
    for prompt, answer in _spec_tokens(case, cfg, seed):
        h, S = _FORWARD[case["family"]](cfg, w, torch.tensor(prompt + answer, device=DEV))
        hidden.append(h)
        states.append(S)
    rows = torch.stack([hidden[r][at + i] for now in _schedule(case) for r, at, _, want in now for i in want])
    head = w["embed"] if case["family"] == "vetevik" else w["head"]
    return {"logits": rows @ head.T * cfg.logit_scale, "states": [torch.stack(s) for s in zip(*states)]}


# --------------------------------------------------------------------------- what is asked of this file
def prepare(case, seed):
    with torch.no_grad():
        return _prepare_dense(case, seed) if case["kind"] == "generate" else _prepare_spec(case, seed)


def run(state):
    return _run_dense(state) if state["kind"] == "generate" else _run_spec(state)


def exact(case, seed):
    with torch.no_grad():
        return _exact_dense(case, seed) if case["kind"] == "generate" else _exact_spec(case, seed)


def _span(first, n):
    """Sum of the positions' key counts over ``n`` tokens from position ``first``."""
    return n * first + n * (n + 1) / 2


def work(case):
    return _work_dense(case) if case["kind"] == "generate" else _work_spec(case)


def _work_dense(case):
    """Every token's projections once; weights once for the prompts and once per decode step (each step needs the token
    before it); the keys and values that a decode step attends to; logits of the sampled rows."""
    cfg = _dense_config(case)
    lens, new, B = _lengths(case, case["batch"]), case["new"], case["batch"]
    per_layer = sum(math.prod(s) for n, s in _dense_shapes(cfg).items() if n.startswith("layers.0.") and len(s) == 2)
    layer, head = per_layer * cfg.num_layers, cfg.vocab_size * cfg.hidden_size
    tokens = sum(n + new - 1 for n in lens)
    pairs = sum(_span(0, n + new - 1) for n in lens)
    flops = 2.0 * layer * tokens + 4.0 * cfg.num_layers * cfg.q_size * pairs + 2.0 * head * B * new
    wb = 2 if case["mode"] in ("bf16", "fp16") else 1
    kv = 4.0 * cfg.num_layers * cfg.kv_size
    reads = sum(_span(n, new - 1) for n in lens)
    return {"bytes": new * (layer * wb + 2.0 * head) + kv * (reads + tokens), "flops": flops}


def _work_spec(case):
    """Per step: every projection of the step's tokens, the experts that they can choose, the attention that each
    layer's mask leaves, the state read and written, the wanted rows' logits."""
    cfg = _spec_config(case)
    b = 4 if case["dtype"] == "fp32" else 2
    shapes = _spec_shapes(case["family"], cfg)
    W, V = cfg.hidden_size, cfg.vocab_size
    bytes_, flops = 0.0, 0.0
    dense = sum(math.prod(s) for n, s in shapes.items() if n.startswith("l") and len(s) == 2 and ".mlp.e" not in n)
    for now in _schedule(case):
        T = sum(n for _, _, n, _ in now)
        bytes_ += dense * b + T * W * b
        flops += 2.0 * dense * T
        for l in cfg.layer_specs:
            m = l.moe
            if m is not None:
                per = (3 if m.glu else 2) * m.ff * W
                flops += 2.0 * per * m.top * T
                bytes_ += per * min(m.experts, m.top * T) * b
            rec = l.ssd or l.delta or l.gla
            if rec is not None:
                cells = rec.heads * rec.vdim * (rec.state if l.ssd else rec.dim)
                flops += (8.0 if l.delta else 6.0) * cells * T
                bytes_ += 8.0 * cells * len(now)
            a = l.attn or l.latent or l.chunk_attn
            if a is not None:
                reach = getattr(a, "window", None) or getattr(a, "chunk", None)
                row = a.cache_dim if l.latent else a.kv_heads * (a.dim + (0 if l.chunk_attn else a.vdim))
                qk = a.dim + a.rot_dim if l.latent else a.dim
                for _, at, n, _ in now:
                    pairs = _span(at, n) if not reach else min(_span(at, n), float(n) * reach)
                    flops += 2.0 * a.heads * (qk + a.vdim) * pairs
                    bytes_ += row * b * min(at + n, reach + n if reach else at + n)
        want = sum(len(e[3]) for e in now)
        if want:
            flops += 2.0 * V * W * want
            bytes_ += V * W * b + 4.0 * V * want
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """The outputs' errors against ``exact`` are 0.003-0.013 (bf16), 0.001 (fp16), 0.02-0.037 (LLM.int8, W8A8: mostly the
    int8 activations, which two implementations round alike but for near-ties) and up to 3e-6 (fp32)."""
    if case["kind"] == "trace" and case["dtype"] == "fp32":
        return {"rel": 1.2e-5}
    return {"rel": 0.004 if case["kind"] == "generate" and case["mode"] == "fp16" else 0.03}
