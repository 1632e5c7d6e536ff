"""Which LM heads of few rows go by the general kernel's small tiles."""
import pytest


@pytest.mark.parametrize("m,n,k,small", [
    (1, 32000, 4096, True), (32, 32000, 2048, True), (32, 128256, 4096, True), (16, 50432, 3072, True), (1, 16384, 512, True),
    (0, 32000, 4096, False), (33, 32000, 4096, False), (1, 8192, 4096, False), (1, 16376, 512, False), (32, 18432, 3072, False),
    (16, 50432, 5120, False), (32, 50257, 1024, False), (1, 2048, 2048, False)])
def test_small_tiles_where_they_are_the_faster(m, n, k, small):
    from kgs.serve.model import head_on_small_tiles

    assert head_on_small_tiles(m, n, k) == small
