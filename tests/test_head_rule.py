"""Which LM heads of few rows go by the general kernel's small tiles, and which gate|up projections by the gate kernel."""
import pytest


@pytest.mark.parametrize("m,n,k,small", [
    (1, 32000, 4096, True), (32, 32000, 2048, True), (32, 128256, 4096, True), (16, 50432, 3072, True), (1, 16384, 512, True),
    (0, 32000, 4096, False), (33, 32000, 4096, False), (1, 8192, 4096, False), (1, 16376, 512, False), (32, 18432, 3072, False),
    (16, 50432, 5120, False), (32, 50257, 1024, False), (1, 2048, 2048, False)])
def test_small_tiles_where_they_are_the_faster(m, n, k, small):
    from kgs.serve.model import head_on_small_tiles

    assert head_on_small_tiles(m, n, k) == small


@pytest.mark.parametrize("m,n,k,route", [
    (39, 2048, 3328, None), (104, 2048, 6912, None), (59, 2304, 1280, (32, 1, 64)), (40, 16384, 4736, (32, 1, 64)), (33, 25856, 1536, (32, 1, 64)),
    (40, 22528, 8064, (128, 1, 128)), (56, 23808, 3840, (128, 1, 128)), (100, 16384, 2048, (32, 1, 128)), (8, 2048, 1024, (32, 1, 64))])
def test_gate_kernel_where_it_is_the_faster(m, n, k, route):
    from kgs.serve.model import gate_up_route

    assert gate_up_route(m, n, k) == route
