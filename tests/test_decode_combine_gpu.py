"""Decode attention over key splits (attn_decode.hip decode_combine_few_kernel up to 4 and 8 splits, decode_combine_kernel):
split counts around those, around the 32 that are read together and the 128 whose weights meet in LDS at once, rows whose
later splits hold no keys."""
import math

import pytest
import torch

from edgellm import ops
from edgellm.ops import _ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,Hq,Hkv", [(64, 4, 1), (128, 2, 2), (80, 2, 1), (256, 2, 1)])
@pytest.mark.parametrize("splits", [2, 3, 4, 5, 8, 9, 31, 32, 33, 64, 65, 128, 129])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_split_counts(D, Hq, Hkv, splits, dt):
    S = splits * 256                                         # 256 keys per split for so few heads
    g = torch.Generator(device="cuda").manual_seed(splits)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g).to(dt)
    q, k, v = r(3, Hq, D), r(3, Hkv, S, D), r(3, Hkv, S, D)
    lens = torch.tensor([S, 1, S - 255], device="cuda", dtype=torch.int32)
    scale = 1 / math.sqrt(D)
    out = ops.ext().decode_attn(q, k, v, lens, scale, S).float()
    ref = _ref.decode_attention(q.float(), k.float(), v.float(), lens, scale)
    mag = _ref.decode_attention(q.float(), k.float(), v.float().abs(), lens, scale)
    # weights, partial sums and scores are fp32; the result is rounded to dt, the weights at most to dt
    eps = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11
    assert ((out - ref).abs() <= eps * (ref.abs() + mag) + 1e-4 * mag + 1e-6).all()
