"""The hashed embedding, the kept previous token and the first input convolution of a one-token step in one launch (postnorm.hip),
bit for bit against the separate ops: slots out of order, sequence starts and stale tails, widths beside a workgroup's, and the
forms that stay apart."""
import pytest
import torch

import edgellm.ops.seqmix as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("W,taps", [(4, 4), (1024, 4), (1028, 4), (2052, 4), (10, 4), (64, 3)])
@pytest.mark.parametrize("seqs", [[(0, 0, 1)], [(5, 1, 1), (2, 9, 1), (0, 0, 1), (3, 2, 1), (1, 3, 1)], [(1, 4, 2), (0, 7, 1)]])
def test_one_launch(cuda, dt, W, taps, seqs, monkeypatch):
    g = torch.Generator().manual_seed(W)
    V, B, T = 33, 13, sum(n for _, _, n in seqs)
    meta = S.RaggedMeta.build(seqs, torch.zeros(6, 1, dtype=torch.int32, device="cuda"), 64, torch.device("cuda"))
    table, big = (torch.randn(n, W, generator=g).to(dt).cuda() for n in (V, B + 1))
    w, state = (torch.randn(W, taps, generator=g) * 0.5).cuda(), torch.randn(6, taps - 1, W, generator=g).cuda()
    state[0] = float("nan")                                  # what an earlier request left in a slot that starts anew
    prev = torch.randint(0, V, (6,), generator=g).cuda()
    ids = torch.randint(-2, V + 2, (T,), generator=g).cuda()
    if len(seqs) == 2:
        state[0] = 1.0
    p2, s2 = prev.clone(), state.clone()
    joined, ran = S._ext().sm_embed_bigram_tap4, []
    monkeypatch.setattr(S._ext(), "sm_embed_bigram_tap4", lambda *a: ran.append(joined(*a)) or ran[-1])
    x, h = S.embedding_bigram_canon(ids, meta, table, big, prev, B, 3, 11, w, state, dt)
    one = all(n == 1 for _, _, n in seqs)                    # where the op tries the launch, and the sizes that it must take
    assert len(ran) == one and (not one or (ran[0] is not None) == (W % 4 == 0 and taps == 4))
    want = S.embedding_bigram(ids, meta, table, big, p2, B, 3, 11)
    assert torch.equal(x, want) and torch.equal(prev, p2)
    assert torch.equal(h, S.canon_conv(want, w, s2, meta, dt)) and torch.equal(state.nan_to_num(7.0), s2.nan_to_num(7.0))


def test_a_portion_without_a_token_keeps_its_previous_one(cuda):
    """It has no last token to read, in front of the step's first or another sequence's."""
    g, V, B, W = torch.Generator().manual_seed(0), 33, 13, 64
    seqs = [(2, 5, 0), (0, 3, 4), (3, 9, 0), (1, 0, 2)]
    meta = S.RaggedMeta.build(seqs, torch.zeros(4, 1, dtype=torch.int32, device="cuda"), 64, torch.device("cuda"))
    table, big = (torch.randn(n, W, generator=g).cuda() for n in (V, B + 1))
    prev, ids = torch.tensor([7, 8, 9, 10]).cuda(), torch.randint(0, V, (6,), generator=g).cuda()
    S.embedding_bigram(ids, meta, table, big, prev, B, 3, 11)
    assert prev.tolist() == [int(ids[3]), int(ids[5]), 9, 10]
