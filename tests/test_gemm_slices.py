"""Which products the general GEMM runs in K slices: by sizes alone, so the scratch that it asks
for tells, with or without a GPU."""
import pytest

torch = pytest.importorskip("torch")


def slices(m, n, k):
    from kgs.ops import _lib

    return int(_lib.lib().kgs_gemm_bf16_nt_scratch(m, n, k)) / (m * ((n + 7) // 8 * 8))


@pytest.mark.parametrize("m,n,k", [(512, 4096, 4096), (496, 4096, 4096), (1024, 1832, 4096), (622, 3072, 4096), (512, 8192, 11008),
                                   (1321, 5120, 14336)])
def test_few_large_tiles_over_a_long_sum_are_sliced(m, n, k):
    """Unsliced these leave a third to half of the CUs idle and take 7 to 30 % longer."""
    assert slices(m, n, k) >= 2


@pytest.mark.parametrize("m,n,k", [(1024, 1024, 3072), (512, 2048, 3072), (413, 2048, 3072), (128, 2048, 2048), (1024, 256, 2048)])
def test_small_tiles_stay_whole(m, n, k):
    """64x64 tiles fill the chip there; slices of larger ones take up to 30 % longer."""
    assert slices(m, n, k) == 0


def test_slices_keep_512_of_the_sum():
    for m in (33, 300, 512):
        for n in (128, 1000, 4096):
            for k in range(128, 16384, 1160):
                assert slices(m, n, k) <= k // 512
