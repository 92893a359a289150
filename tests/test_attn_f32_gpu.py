"""fp32 prompt attention on the matrix cores (attn_f32.hip) against the same op on the CPU: every head size, heads of a kv head 4, 2
and 1 at a time, portions beside 16 and 64 rows, two and four groups of key tiles, windows, kept first tokens, pooled blocks, chunks,
caps, slopes, sinks, distance biases, gates and result views; numbers that are not finite behind a query's mask."""
import pytest
import torch

import edgellm.ops.seqmix as S

pytestmark = pytest.mark.gpu
PAGE = 64
_form = 0


def _check(seqs, H, G, D, Dv, run, pool=0, latent=False, seed=0, spoil=None):
    """``seqs``: (tokens held, tokens brought) per sequence."""
    if _form == 2 + 32 and max(D, Dv) > 64:
        pytest.skip("four groups of key tiles: rows of up to 64 numbers")
    g = torch.Generator().manual_seed(seed)
    per = max(a + b for a, b in seqs) // PAGE + 1
    pages, T = per * len(seqs), sum(b for _, b in seqs)
    table = torch.randperm(pages, generator=g).view(len(seqs), per).int()
    k = torch.randn(pages, PAGE, G, D, generator=g)
    v = k[..., :Dv] if latent else torch.randn(pages, PAGE, G, Dv, generator=g)
    q = torch.randn(T, H, D, generator=g)
    kb = torch.randn(pages, PAGE // pool, G, D, generator=g) if pool else None
    vb = torch.randn(pages, PAGE // pool, G, Dv, generator=g) if pool else None

    def on(dev):
        c = lambda t: None if t is None else t.to(dev)
        kd, vd = c(k), c(v)
        if spoil and dev == "cuda":                          # (the CPU's op multiplies what is not seen by 0)
            spoil(kd, vd, table)
        m = S.RaggedMeta.build([(i, a, b) for i, (a, b) in enumerate(seqs)], table.to(dev), PAGE, dev)
        return run(c(q), kd, kd[..., :Dv] if latent else vd, c(kb), c(vb), m, c)
    got, ref = on("cuda").cpu(), on("cpu")
    # fp32 sums under weights of sum 1 over values of about 1, on both sides; a key left out or taken twice among some hundred changes 1 / 300
    ok = got.isfinite()
    assert ok.all() or spoil
    assert ((got - ref).abs() <= 2.0 ** -17 * ref.abs() + 2.0 ** -17)[ok].all(), (got - ref).abs()[ok].max()
    return got


@pytest.fixture(autouse=True, params=[4 + 16, 2 + 16, 2 + 32, 0])
def form(request, monkeypatch):
    """Query-row waves and groups of key tiles, and the rule's choice.  A form that is asked for runs, or the op raises."""
    global _form
    _form, tiles = request.param, S._portions
    if request.param:
        monkeypatch.setattr(S, "_portions", lambda *a: (tiles(*a)[0], -request.param))


SIZES = [(32, 32), (64, 64), (96, 96), (128, 128), (64, 128), (128, 64)]


@pytest.mark.parametrize("H,G", [(8, 2), (4, 2), (3, 3)])
@pytest.mark.parametrize("D,Dv", SIZES)
@pytest.mark.parametrize("seqs", [[(0, 16)], [(0, 65), (130, 17), (63, 1)], [(70, 300), (0, 128)]])
def test_plain(H, G, D, Dv, seqs):
    T = sum(b for _, b in seqs)
    gate = torch.randn(T, H, generator=torch.Generator().manual_seed(1))
    _check(seqs, H, G, D, Dv, lambda q, k, v, kb, vb, m, on: S.window_pool_attention(
        q, on(gate), k, v, None, None, m, D ** -0.5, None, None, on(torch.linspace(-1, 3, H))))


@pytest.mark.parametrize("D,Dv", [(160, 128), (128, 128), (64, 64)])
@pytest.mark.parametrize("window", [None, 70])
def test_latent(D, Dv, window):
    _check([(5, 200), (0, 40)], 16, 1, D, Dv, lambda q, k, v, kb, vb, m, on: S.window_pool_attention(
        q, None, k, v, None, None, m, D ** -0.5, window, None), latent=True)


@pytest.mark.parametrize("window,pool,keep", [(100, 4, 0), (64, 16, 0), (33, 0, 20), (64, 0, 70), (300, 1, 0), (512, 64, 0)])
@pytest.mark.parametrize("seqs", [[(0, 400)], [(190, 130), (0, 16)], [(0, 20)] * 40])
def test_windows(window, pool, keep, seqs):
    _check(seqs, 8, 2, 64, 64, lambda q, k, v, kb, vb, m, on: S.window_pool_attention(
        q, None, k, v, kb, vb, m, 0.125, window, pool or None, None, keep), pool=pool)


@pytest.mark.parametrize("chunk,cap,slopes", [(None, 5.0, False), (64, None, True), (50, 2.0, True)])
@pytest.mark.parametrize("D", [32, 64, 96, 128])
def test_chunks(chunk, cap, slopes, D):
    gate = torch.randn(245, 8 * D, generator=torch.Generator().manual_seed(2))
    sl = S.distance_slopes(8) if slopes else None
    _check([(30, 200), (0, 45)], 8, 2, D, D, lambda q, k, v, kb, vb, m, on: S.chunk_attention(
        q, on(gate), k, m, 0.125, chunk, cap, on(sl), on(torch.zeros(8))), latent=True)


def test_bias_view_and_many_workgroups():
    """A bias by distance, a result written times a number into a wider matrix, 30 portions."""
    rel = torch.randn(8, 70, generator=torch.Generator().manual_seed(3))

    def run(q, k, v, kb, vb, m, on):
        wide = torch.zeros(q.shape[0], 8 * 64 + 32, dtype=q.dtype, device=q.device)
        S.window_pool_attention(q, None, k, v, None, None, m, 0.1, 200, None, None, 3, on(rel), wide[:, 32:], 0.5)
        assert (wide[:, :32] == 0).all()
        return wide
    _check([(9, 180)] * 30, 8, 8, 64, 64, run)


def test_numbers_that_a_query_does_not_see():
    """Infinities and NaN among later keys, in another sequence's old rows and before the window change no result; a query that sees
    one shows it."""
    def spoil(k, v, table):
        v[table[0, 2], 10] = float("nan")                    # position 138: seen from 138 to 187 through the window
        v[table[0, 0], 5] = float("inf")                     # position 5: up to 54
        v[table[0, 3], 40:] = float("inf")                   # past the last token
        k[table[0, 3], 40:] = float("nan")
    got = _check([(0, 230)], 8, 2, 64, 64, lambda q, k, v, kb, vb, m, on: S.window_pool_attention(
        q, None, k, v, None, None, m, 0.125, 50, None), spoil=spoil)
    bad = ~got.isfinite().all(1)
    assert bad.tolist() == [5 <= t < 55 or 138 <= t < 188 for t in range(230)]


def test_a_form_that_does_not_fit_is_refused():
    """What the tests above rest on: no other kernel stands in for the form that they ask for."""
    if _form == 0:
        pytest.skip("the rule's choice may be another kernel")
    with pytest.raises(RuntimeError, match="form"):
        _check([(0, 40)], 4, 4, 48, 48, lambda q, k, v, kb, vb, m, on: S.window_pool_attention(
            q, None, k, v, None, None, m, 0.125, None, None))
