"""Which steps take the fp32 prompt attention on the matrix cores (attn_f32.hip), by its estimates: steps measured on either side."""
import pytest

from edgellm.ops import seqmix


def plan(H, G, D, Dv, rows, vis, mean, n=1, windowed=False, same=False):
    return seqmix._ext().sm_attention_f32_plan(rows, n, H, G, D, Dv, same, windowed, vis, mean, 0)


@pytest.fixture(autouse=True)
def built():
    if not seqmix.available():
        pytest.skip("extension not built")


# heads, groups, row and value width, rows, keys of the last and of the middle row
@pytest.mark.parametrize("size", [
    (16, 4, 128, 128, 191, 191, 96),            # us, the kernels before / here: 17.1 / 21.2
    (16, 4, 128, 128, 130, 130, 66),            # 15.2 / 21.6
    (2, 1, 128, 128, 449, 449, 225),            # 20.5 / 36.8
    (16, 4, 64, 64, 100, 100, 51),              # 8.8 / 9.2
    (16, 4, 64, 64, 20, 1020, 1010)])           # 16.7 / 30
def test_kept_by_the_kernels_before(size):
    assert plan(*size) == 0


def test_kept_by_the_kernels_before_behind_a_window():
    assert plan(6, 3, 64, 128, 331, 128, 128, windowed=True) == 0                  # 12.0 / 18.7
    assert plan(2, 1, 128, 128, 1077, 128, 120, n=2, windowed=True) == 0           # 20.4 / 22.9


@pytest.mark.parametrize("size", [
    (16, 4, 64, 64, 1024, 512, 256),            # two portions of 512
    (16, 4, 64, 64, 2000, 2000, 1001),          # 342 / 102
    (16, 4, 128, 128, 1000, 1000, 501),         # 205 / 78
    (16, 16, 64, 64, 2000, 2000, 1001)])        # 1115 / 102
def test_taken(size):
    assert plan(*size) > 0


def test_latent_rows_are_taken():
    assert plan(16, 1, 160, 128, 300, 300, 151, same=True) > 0                     # 65 / 26
