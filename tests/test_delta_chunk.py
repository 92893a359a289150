"""The chunked form of the gated delta rule (csrc/seqmix/delta_chunk.hip) against the recurrence in float64."""
import pytest
import torch

import edgellm  # noqa: F401
from edgellm.ops import seqmix

gpu = pytest.mark.gpu


def recurrence(prep, v, S, G, H, N, channel):
    """prep [L, q | k | decay | beta], v [L, H, P], S [H, N, P], all float64."""
    GN, rep, D = G * N, H // G, H * (N if channel else 1)
    q, k = (prep[:, i * GN:(i + 1) * GN].view(-1, G, N).repeat_interleave(rep, 1) for i in (0, 1))
    g, beta = prep[:, 2 * GN:2 * GN + D].view(len(prep), H, -1), prep[:, 2 * GN + D:]
    out = torch.empty_like(v)
    for t in range(len(prep)):
        S = S * g[t][:, :, None]
        w = beta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
        S = S + k[t][:, :, None] * w[:, None, :]
        out[t] = (S * q[t][:, :, None]).sum(1)
    return out, S


def inputs(lens, starts, H, G, N, P, channel, decay, seed=0, keys="random"):
    g = torch.Generator().manual_seed(seed)
    T = sum(lens)
    meta = seqmix.RaggedMeta.build([(len(lens) - 1 - i, st, L) for i, (st, L) in enumerate(zip(starts, lens))],
                                   torch.zeros(len(lens), 4, dtype=torch.int32, device="cuda"), 64, "cuda")
    qkv = torch.nn.functional.silu(torch.randn(T, 2 * G * N + H * P, generator=g)).bfloat16().cuda()
    unit = torch.randn(2, T, G, N, generator=g)
    if keys == "alike":                                # about 0.98 of each other's direction
        unit = torch.nn.functional.normalize(unit, dim=-1) * 0.14 + torch.nn.functional.normalize(torch.randn(G, N, generator=g), dim=-1)
    unit = torch.nn.functional.normalize(unit, dim=-1)
    D = H * (N if channel else 1)
    d = {"weak": 1.0 - 1e-4 * torch.rand(T, D, generator=g), "usual": torch.rand(T, D, generator=g) ** 0.1,
         "none": torch.ones(T, D), "strong": torch.rand(T, D, generator=g) * 1e-3, "mixed": torch.where(torch.rand(T, D, generator=g) < 0.1, 0.0, 0.99)}[decay]
    prep = torch.cat([(unit[0] * N ** -0.5).reshape(T, -1), unit[1].reshape(T, -1), d,
                      (0.97 + 0.03 * torch.rand(T, H, generator=g)) if keys == "alike" else torch.rand(T, H, generator=g)], -1)
    state = torch.randn(len(lens), H, N, P, generator=g)
    return prep.cuda(), qkv, state.cuda(), meta


# fp64 inside; inputs of the outputs' products and the states rounded to fp32 (2^-25 rms 3e-8 each): bound 2e-7
TOL = 2e-7


@gpu
@pytest.mark.parametrize("channel", [True, False])
@pytest.mark.parametrize("decay", ["weak", "usual", "strong", "mixed"])
@pytest.mark.parametrize("lens,starts,H,G,N,P", [
    ((64, 63, 65), (0, 5, 0), 4, 4, 64, 64),          # about one chunk
    ((200, 1, 16), (3, 7, 0), 4, 2, 24, 20),          # odd sizes, shared keys, a decode token and a short portion beside
    ((321,), (0,), 2, 2, 128, 48),                    # 128 channels: two quarters
    ((130, 17), (1, 0), 2, 1, 200, 70)])              # up to 256 channels: four quarters
def test_chunks_against_the_recurrence(lens, starts, H, G, N, P, channel, decay, monkeypatch):
    prep, qkv, state, meta = inputs(lens, starts, H, G, N, P, channel, decay)
    before = state.double().cpu()
    monkeypatch.setattr(seqmix, "DELTA_CHUNK_MIN", 1)
    y = seqmix.delta_rule_scan(prep, qkv, state, meta, H, G, N, P).double().cpu()
    p, v = prep.double().cpu(), qkv[:, 2 * G * N:].double().cpu().view(len(prep), H, P)
    for slot, start, n, off in meta.host:
        S0 = before[slot] if start > 0 else torch.zeros(H, N, P, dtype=torch.float64)
        want, S = recurrence(p[off:off + n], v[off:off + n], S0, G, H, N, channel)
        got = y[off:off + n].view(n, H, P)
        assert (got - want).norm() < TOL * want.norm() and (got - want).abs().max() < 20 * TOL * want.abs().max()
        assert (state[slot].double().cpu() - S).norm() < TOL * S.norm().clamp_min(1e-3)


@gpu
@pytest.mark.parametrize("n,H,G,N,P", [
    (1, 16, 16, 64, 64), (1, 12, 4, 72, 80), (2, 16, 8, 33, 64), (2, 9, 3, 128, 112),    # 4 and 8 columns a workgroup
    (5, 16, 8, 20, 80), (4, 11, 1, 100, 96), (9, 7, 7, 64, 16), (1, 1, 1, 64, 1)])       # 8, 16, 4; heads that do not fill the eight dies
def test_chunks_at_every_split_of_the_columns(n, H, G, N, P, monkeypatch):
    prep, qkv, state, meta = inputs((129, 64, 30, 70, 1, 65, 2, 128, 3)[:n], (5, 0, 1, 0, 3, 0, 0, 2, 1)[:n], H, G, N, P, True, "usual", seed=n)
    before = state.double().cpu()
    monkeypatch.setattr(seqmix, "DELTA_CHUNK_MIN", 1)
    y = seqmix.delta_rule_scan(prep, qkv, state, meta, H, G, N, P).double().cpu()
    p, v = prep.double().cpu(), qkv[:, 2 * G * N:].double().cpu().view(len(prep), H, P)
    for slot, start, length, off in meta.host:
        S0 = before[slot] if start > 0 else torch.zeros(H, N, P, dtype=torch.float64)
        want, S = recurrence(p[off:off + length], v[off:off + length], S0, G, H, N, True)
        assert (y[off:off + length].view(length, H, P) - want).norm() < TOL * want.norm()
        assert (state[slot].double().cpu() - S).norm() < TOL * S.norm().clamp_min(1e-3)


@gpu
@pytest.mark.parametrize("channel", [True, False])
@pytest.mark.parametrize("keys,decay", [("random", "usual"), ("random", "weak"), ("random", "strong"), ("alike", "none"), ("alike", "weak")])
@pytest.mark.parametrize("H,G,N,P", [(4, 2, 64, 64), (2, 2, 128, 64), (2, 1, 200, 70)])
def test_chunks_are_no_further_off_than_the_recurrence_in_fp32(H, G, N, P, channel, keys, decay, monkeypatch):
    """Outputs and states, also with keys that resemble each other, where a chunk's terms cancel."""
    prep, qkv, state, meta = inputs((321, 70), (0, 9), H, G, N, P, channel, decay, 3, keys)
    p, v, off = prep.double().cpu(), qkv[:, 2 * G * N:].double().cpu().view(len(prep), H, P), [(m[3], m[2], m[0], m[1]) for m in meta.host]
    want = [recurrence(p[o:o + n], v[o:o + n], state[s].double().cpu() * (st > 0), G, H, N, channel) for o, n, s, st in off]
    err = []
    for least in (1 << 30, 1):
        monkeypatch.setattr(seqmix, "DELTA_CHUNK_MIN", least)
        S = state.clone()
        y = seqmix.delta_rule_scan(prep, qkv, S, meta, H, G, N, P).double().cpu()
        err.append([(((y[o:o + n].view(n, H, P) - w[0]).norm() / w[0].norm()).item(), ((S[s].double().cpu() - w[1]).norm() / w[1].norm()).item())
                    for (o, n, s, _), w in zip(off, want)])
    steps, chunks = torch.tensor(err[0]), torch.tensor(err[1])
    assert (chunks <= steps).all(), (chunks, steps)


@pytest.mark.parametrize("lens,H,N,least", [
    ((160,), 16, 64, 0), ((300,), 16, 64, 1), ((4096,), 4, 64, 1), ((512,) + (1,) * 5, 16, 64, 128), ((512,) + (1,) * 63, 16, 64, 128),
    ((256,) + (1,) * 255, 16, 64, 0), ((512,) * 8, 16, 64, 0), ((512,) * 8, 4, 64, 1), ((1,) * 40, 16, 64, 0), ((512, 512), 16, 128, 1),
    ((512,) * 32, 16, 128, 0), ((1000, 300, 0, 100), 16, 128, 128), ((160,), 4, 256, 0), ((512,) * 32, 16, 256, 1),
    ((4096,), 16, 257, 0), ((), 16, 64, 0)])
def test_portions_take_the_shorter_form(lens, H, N, least):
    """The length from which on portions run over chunks (1: all of them do)."""
    assert seqmix.delta_chunks_from(lens, H, N, N) == least


@pytest.mark.parametrize("chunks,room,parts", [
    ([64], 64, (64, 64)), ([64], 63, (32, 32)), ([9], 1, (1, 1)), ([8, 3], 9, (4, 7)), ([8, 3], 11, (8, 11)), ([2, 2, 2], 2, (0, 0)),
    ([1, 1, 1], 3, (1, 3)), ([], 5, (0, 0)), ([7], 0, (0, 0))])
def test_portions_run_in_parts_that_fit_the_scratch(chunks, room, parts):
    assert seqmix.delta_parts(chunks, room) == parts


@gpu
@pytest.mark.parametrize("channel,H,N,P", [(True, 4, 64, 48), (False, 2, 128, 64), (True, 2, 200, 70)])
@pytest.mark.parametrize("room", [3, 5, 7, 0])
def test_parts_carry_the_state(channel, H, N, P, room, monkeypatch):
    """Portions of several lengths in parts of one, two and four chunks each, and in none (token by token)."""
    monkeypatch.setattr(seqmix, "DELTA_CHUNK_MIN", 100)
    prep, qkv, state, meta = inputs((330, 20, 130, 500), (0, 3, 5, 64), H, 2, N, P, channel, "usual", 5)
    S, Sw = state.clone(), state.clone()
    whole = seqmix.delta_rule_scan(prep, qkv, Sw, meta, H, 2, N, P)
    monkeypatch.setattr(seqmix, "DELTA_SCRATCH_BYTES", room * 4 * seqmix._ext().sm_delta_chunk_floats(1, H, N, P))
    y = seqmix.delta_rule_scan(prep, qkv, S, meta, H, 2, N, P)
    # the state is rounded to fp32 between parts (2^-25 rms 3e-8 of its size each time); room 0: the recurrence in fp32
    tol = 2e-7 if room else 6e-7
    assert (y - whole).norm() < tol * whole.norm() and (S - Sw).norm() < tol * Sw.norm()
    assert not torch.equal(y, whole) and torch.equal(y[330:350], whole[330:350])


@gpu
@pytest.mark.parametrize("channel", [True, False])
def test_long_and_short_portions_of_one_step(channel, monkeypatch):
    """Long ones over chunks, the others token by token, each with its own slot; portions at the line itself."""
    lens, starts, H, G, N, P = (130, 1, 64, 16, 63, 200), (3, 700, 0, 0, 9, 1), 4, 2, 64, 48
    prep, qkv, state, meta = inputs(lens, starts, H, G, N, P, channel, "usual", 4)
    res = []
    for least in (64, 1, 1 << 30):
        monkeypatch.setattr(seqmix, "DELTA_CHUNK_MIN", least)
        S = state.clone()
        res.append((seqmix.delta_rule_scan(prep, qkv, S, meta, H, G, N, P), S))
    (y, S), (yc, Sc), (yt, St) = res
    for slot, _, n, off in meta.host:
        w, Sw = (yc, Sc) if n >= 64 else (yt, St)
        assert torch.equal(y[off:off + n], w[off:off + n]) and torch.equal(S[slot], Sw[slot])


@gpu
def test_long_portions_run_over_chunks_and_fp32_steps_stay_token_by_token(monkeypatch):
    prep, qkv, state, meta = inputs((300, 40), (0, 9), 2, 2, 64, 32, True, "usual", 1)
    a, b = state.clone(), state.clone()
    chunks = seqmix.delta_rule_scan(prep, qkv, a, meta, 2, 2, 64, 32)
    monkeypatch.setattr(seqmix, "DELTA_CHUNK_MIN", 1 << 30)
    steps = seqmix.delta_rule_scan(prep, qkv, b, meta, 2, 2, 64, 32)
    assert not torch.equal(chunks, steps) and torch.allclose(chunks, steps, atol=1e-5) and torch.allclose(a, b, atol=1e-5)
    monkeypatch.undo()
    c, d = state.clone(), state.clone()
    y = seqmix.delta_rule_scan(prep, qkv.float(), c, meta, 2, 2, 64, 32)
    monkeypatch.setattr(seqmix, "DELTA_CHUNK_MIN", 1 << 30)
    assert torch.equal(y, seqmix.delta_rule_scan(prep, qkv.float(), d, meta, 2, 2, 64, 32)) and torch.equal(c, d)


@gpu
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_a_value_that_is_not_finite_reaches_no_earlier_token(bad, monkeypatch):
    monkeypatch.setattr(seqmix, "DELTA_CHUNK_MIN", 1)
    prep, qkv, state, meta = inputs((100, 70), (0, 0), 2, 2, 64, 32, True, "usual", 2)
    clean = seqmix.delta_rule_scan(prep, qkv, state.clone(), meta, 2, 2, 64, 32)
    qkv[75, -3] = bad                                  # a value of head 1, in the middle of a block
    y = seqmix.delta_rule_scan(prep, qkv, state.clone(), meta, 2, 2, 64, 32)
    assert torch.allclose(y[:75], clean[:75], atol=1e-6) and torch.allclose(y[100:], clean[100:], atol=1e-6)
    assert torch.allclose(y[75:100, :32], clean[75:100, :32], atol=1e-6) and not y[75, -3].isfinite()
