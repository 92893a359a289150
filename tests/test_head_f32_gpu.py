"""The output projection that stores fp32 (up to 16 bf16 rows) against the same GEMV's bf16 rows widened, bit for bit: the tiles form, two
and four tiles a workgroup, a last group that is not full; and calls that it leaves to the projection itself."""
import pytest
import torch

from edgellm.models.layers import Linear

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(16, 64), (320, 192), (8192, 4096), (10000, 256), (16384, 128), (16400, 1024), (32000, 1024)])
@pytest.mark.parametrize("M", [1, 4, 5, 8, 9, 12, 16])
@torch.no_grad()
def test_rows(N, K, M):
    g = torch.Generator(device="cuda").manual_seed(N + M)
    lin = Linear(K, N, False, torch.bfloat16, torch.device("cuda"))
    lin.weight.copy_(torch.randn(N, K, generator=g, device="cuda"))
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    y = lin.forward_f32(x)
    assert y.dtype == torch.float32 and torch.equal(y, lin(x).float())


@torch.no_grad()
def test_not_taken():
    lin = Linear(128, 64, False, torch.bfloat16, torch.device("cuda"))
    assert lin.forward_f32(torch.zeros(17, 128, device="cuda", dtype=torch.bfloat16)) is None
    with torch.enable_grad():
        x = torch.zeros(2, 128, device="cuda", dtype=torch.bfloat16, requires_grad=True)
        assert lin.forward_f32(x) is None
    hook = lin.register_forward_hook(lambda *a: None)
    assert lin.forward_f32(torch.zeros(2, 128, device="cuda", dtype=torch.bfloat16)) is None
    hook.remove()
