"""Prompt attention over latent rows on the matrix cores (latent_mfma.hip) against the same op in fp32 on the CPU, over the
head sizes it takes: portions around its 32-query and 64-key tiles, head counts that fill a workgroup's eight waves and ones
that do not, windows, cached keys before the portion, wide cache rows, result rows of every alignment."""
import pytest
import torch

import edgellm.ops.seqmix as S

pytestmark = pytest.mark.gpu

DIMS = [(128, 96), (160, 128), (192, 128), (320, 256)]
STEPS = {  # (slot, cached, new) per sequence
    "one": [(0, 0, 16)],
    "edges": [(0, 0, 31), (2, 64, 32), (1, 33, 33), (3, 127, 1), (5, 1, 63), (4, 0, 65)],
    "long": [(1, 130, 257), (0, 0, 129)],
}


def _case(seqs, H, D, Dv, wide, seed):
    g = torch.Generator().manual_seed(seed)
    slots, pages = max(s for s, _, _ in seqs) + 1, [(a + n + 63) // 64 for _, a, n in seqs]
    perm, tab, k = torch.randperm(sum(pages) + 1, generator=g).int(), torch.zeros(slots, max(pages), dtype=torch.int32), 0
    for (s, _, _), c in zip(seqs, pages):
        tab[s, :c] = perm[k:k + c]
        k += c
    T = sum(n for _, _, n in seqs)
    rows = torch.randn(sum(pages) + 1, 64, 1, D + wide, generator=g).bfloat16()
    return tab, rows, torch.randn(T, H, D, generator=g).bfloat16(), torch.randn(T, H, generator=g).bfloat16()


def _check(seqs, H, D, Dv, window=None, wide=0, gated=True, out=None, out_scale=1.0, seed=0):
    dev = torch.device("cuda:0")
    tab, rows, q, gate = _case(seqs, H, D, Dv, wide, seed)

    def run(d, dt, v_abs=False):
        meta = S.RaggedMeta.build(seqs, tab.to(d), 64, d)
        kp = rows.to(d, dt)[..., :D]
        vp = (kp.abs() if v_abs else kp)[..., :Dv]
        return S.window_pool_attention(q.to(d, dt), gate.to(d, dt) if gated else None, kp, vp, None, None, meta, D ** -0.5,
                                       window, None, out=out if d == dev else None, out_scale=out_scale)

    got = run(dev, torch.bfloat16).float().cpu()
    ref, mag = run(torch.device("cpu"), torch.float32), run(torch.device("cpu"), torch.float32, True)
    # weights and result are rounded to bf16 (8 significant bits: 2^-8 of each at most); fp32 scores move a weight far less
    bound = 2.0 ** -8 * mag.abs() + 2.0 ** -8 * ref.abs() + 1e-4 * mag.abs() + 1e-6
    over = ((got - ref).abs() / bound).max()
    assert over <= 1.0, over


@pytest.mark.parametrize("D,Dv", DIMS)
@pytest.mark.parametrize("H", [1, 2, 3, 4, 6, 8, 12, 16])
@pytest.mark.parametrize("step,window", [("one", None), ("edges", None), ("edges", 30), ("long", 1), ("long", 64), ("long", 100),
                                         ("long", None)])
def test_latent_prompt(D, Dv, H, step, window):
    _check(STEPS[step], H, D, Dv, window, seed=H)


@pytest.mark.parametrize("D,Dv", DIMS)
@pytest.mark.parametrize("pad,first,lines", [(0, 0, True), (8, 0, True), (16, 8, True), (24, 16, True), (8, 4, False), (4, 0, False),
                                             (3, 1, False), (9, 8, False)])
def test_latent_prompt_rows(D, Dv, pad, first, lines):
    """Wide cache rows, no gate, result rows in a wider matrix: whole-line stores where its rows and its start are whole 16
    bytes (also with room on either side), number by number elsewhere; the columns beside the slice stay."""
    H, T = 8, sum(n for _, _, n in STEPS["edges"])
    wide = torch.full((T, H * Dv + pad), 7.0, device="cuda:0").bfloat16()
    out = wide[:, first:first + H * Dv]
    assert (out.stride(0) % 8 == 0 and out.data_ptr() % 16 == 0) == lines
    _check(STEPS["edges"], H, D, Dv, 50, wide=40, gated=False, out=out, out_scale=0.5)
    assert (wide[:, :first] == 7).all() and (wide[:, first + H * Dv:] == 7).all()


def test_latent_prompt_of_two_million_tokens():
    """More query tiles than a grid's second dimension may hold; with a window of one token the result is the token's value."""
    H, D, Dv, T = 8, 128, 96, (1 << 21) + 77
    g = torch.Generator(device="cuda:0").manual_seed(0)
    rows = torch.randn((T + 63) // 64, 64, 1, D, generator=g, device="cuda:0", dtype=torch.bfloat16)
    q = torch.randn(T, H, D, generator=g, device="cuda:0", dtype=torch.bfloat16)
    meta = S.RaggedMeta.build([(0, 0, T)], torch.arange(rows.shape[0], dtype=torch.int32, device="cuda:0")[None], 64, "cuda:0")
    out = S.window_pool_attention(q, None, rows, rows[..., :Dv], None, None, meta, D ** -0.5, 1, None)
    want = rows.view(-1, D)[:T, :Dv]
    for h in range(H):
        assert torch.equal(out.view(T, H, Dv)[:, h], want)
