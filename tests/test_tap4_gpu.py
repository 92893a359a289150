"""Four-tap convolutions over ragged rows (tap4.h) against the same ops on the CPU, results and kept tails: portions shorter
than, as long as and longer than the tail, at a sequence's start and behind one, both row blocks (one token below 512 rows,
four from there), channel counts beside a workgroup's, and the forms that stay with the general kernels (other taps, columns
that are not a multiple of 16 bytes)."""
import pytest
import torch

import edgellm.ops.seqmix as S

pytestmark = pytest.mark.gpu

STEPS = {
    "decode": [(2, 9, 1), (0, 0, 1), (5, 1, 1), (1, 2, 1), (3, 3, 1)],
    "short": [(1, 0, 1), (0, 1, 2), (4, 2, 3), (2, 0, 4), (5, 700, 5), (3, 0, 2)],
    "below": [(0, 5, 255), (3, 0, 256)],
    "at": [(0, 0, 1), (3, 2, 510), (1, 1, 1)],
    "above": [(2, 3, 513), (1, 0, 3), (0, 2, 1), (4, 6, 254)],
}


def _run(op, seqs, dev, dt, out, C, taps, c0, seed):
    g = torch.Generator().manual_seed(seed)
    T = sum(n for _, _, n in seqs)
    meta = S.RaggedMeta.build(seqs, torch.zeros(6, 1, dtype=torch.int32, device=dev), 64, dev)
    u, w, b = torch.randn(T, c0 + C + 8, generator=g), torch.randn(C, taps, generator=g) * 0.5, torch.randn(C, generator=g)
    state = torch.randn(6, taps - 1, C, generator=g)
    for slot, start, _ in seqs:                              # as an earlier portion leaves it: zero before the first token
        state[slot, :max(taps - 1 - start, 0)] = 0 if start else 1
    if op == "silu":
        u, state = u.to(dt).to(dev, out), state.to(dt).to(dev, out)
        return S.conv_silu(u, c0, C, w.to(dev), b.to(dev), state, meta), state
    x, state = u[:, :C].contiguous().to(dev), state.to(dev)
    return S.canon_conv(x, w.to(dev), state, meta, out), state


@pytest.mark.parametrize("step", list(STEPS))
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("op,C,taps,c0", [("silu", 8, 4, 0), ("silu", 2056, 4, 16), ("silu", 1040, 4, 4), ("silu", 20, 4, 8),
                                          ("silu", 64, 3, 8), ("plain", 4, 4, 0), ("plain", 1028, 4, 0), ("plain", 1030, 4, 0),
                                          ("plain", 64, 6, 0)])
def test_tap4(step, dt, op, C, taps, c0):
    got, kept = _run(op, STEPS[step], torch.device("cuda:0"), dt, dt, C, taps, c0, C)
    ref, tail = _run(op, STEPS[step], torch.device("cpu"), dt, torch.float32, C, taps, c0, C)
    assert torch.equal(kept.cpu().float(), tail)                     # inputs as they came
    # a handful of fp32 products and sums of size <= 20 (2^-24 each), silu's expf, then one rounding to the output type
    tol = 1e-5 + (2.0 ** -8 if dt == torch.bfloat16 else 1e-5) * ref.abs()
    assert ((got.cpu().float() - ref).abs() <= tol).all()


@pytest.mark.parametrize("rows", [30, 600])
@pytest.mark.parametrize("op,dt", [("silu", torch.bfloat16), ("silu", torch.float32), ("plain", torch.float32)])
def test_portions_without_a_token(op, dt, rows):
    """They clear what lies in front of their sequence's start, keep the rest of the tail, and change nothing for the others."""
    dev, C = torch.device("cuda:0"), 1032
    full, empty = [(0, 4, rows), (4, 0, 2)], [(2, 0, 0), (0, 4, rows), (1, 1, 0), (5, 9, 0), (4, 0, 2), (3, 2, 0)]
    g = torch.Generator().manual_seed(rows)
    u, w, b = torch.randn(rows + 2, C, generator=g).to(dt).to(dev), torch.randn(C, 4, generator=g).to(dev), torch.randn(C, generator=g).to(dev)
    kept = torch.randn(6, 3, C, generator=g).to(dt).to(dev)
    res = []
    for seqs in (full, empty):
        meta, state = S.RaggedMeta.build(seqs, torch.zeros(6, 1, dtype=torch.int32, device=dev), 64, dev), kept.clone()
        y = S.conv_silu(u, 0, C, w, b, state, meta) if op == "silu" else S.canon_conv(u, w, state, meta, dt)
        res.append((y, state))
    assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1][[0, 4]], res[1][1][[0, 4]])
    state = res[1][1]
    assert not state[2].any() and not state[1, :2].any() and not state[3, 0].any()
    assert torch.equal(state[5], kept[5]) and torch.equal(state[1, 2], kept[1, 2]) and torch.equal(state[3, 1:], kept[3, 1:])
