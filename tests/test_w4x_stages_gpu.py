"""Four-wave tiles of 128 rows or columns, which run on three and four LDS stages with one barrier a K-step, against what runs on two: 256x256 tiles, in slices and
gated, and the gate of the product's rounded halves. K-tiles a slice: fewer than the stages, as many, one round of them and more."""
import pytest
import torch

from kgs.ops.activation import Gate
from kgs.ops.gemm import gemm_nt_w4x, gemm_nt_w4x_partials, gemm_nt_w4x_swiglu, pack_w4x_weight
from kgs.ops.transformer import silu_mul

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("own_rng")]
TILES = ((128, 128), (256, 128), (128, 256))


def _operands(m, n, k):
    return (torch.rand(m, k, device="cuda") * 2 - 1).bfloat16(), ((torch.rand(n, k, device="cuda") * 2 - 1) * k ** -0.5).bfloat16()


@pytest.mark.parametrize("bm,bn", TILES)
@pytest.mark.parametrize("ks", (128, 256, 384, 512, 640))
@pytest.mark.parametrize("m,nslice", ((72, 2), (128, 3), (200, 4)))
def test_slices_keep_the_bits_of_two_stages(bm, bn, ks, m, nslice):
    a, w = _operands(m, 512, ks * nslice)
    want = gemm_nt_w4x_partials(a, w, 256, nslice, bm=256, private=True)
    total = gemm_nt_w4x(a, w, bn=256, nslice=nslice, bm=256)
    for b in (w, pack_w4x_weight(w, bn)):
        for nt in (False, True):
            assert torch.equal(gemm_nt_w4x_partials(a, b, bn, nslice, bm=bm, nt_weights=nt, private=True), want)
            assert torch.equal(gemm_nt_w4x(a, b, bn=bn, nslice=nslice, bm=bm, nt_weights=nt), total)


@pytest.mark.parametrize("bm,bn", TILES)
@pytest.mark.parametrize("k", (128, 256, 384, 512, 640, 1152))
@pytest.mark.parametrize("m", (72, 200))
def test_gated_tiles_keep_the_bits_of_two_stages(bm, bn, k, m):
    a, w = _operands(m, 1024, k)
    want = silu_mul(gemm_nt_w4x(a, w, bn=256, bm=256))  # the product's halves, rounded, and their gate
    assert torch.equal(gemm_nt_w4x_swiglu(a, w, bn=256, bm=256), want)
    for b in (w, pack_w4x_weight(w, bn, swiglu=True)):
        for nt in (False, True):
            assert torch.equal(gemm_nt_w4x_swiglu(a, b, bn=bn, bm=bm, nt_weights=nt), want)
    for act in ("gelu_tanh", Gate("clamped", 0.4)):
        want = gemm_nt_w4x_swiglu(a, w, bn=256, bm=256, act=act)
        for nt in (False, True):
            assert torch.equal(gemm_nt_w4x_swiglu(a, w, bn=bn, bm=bm, nt_weights=nt, act=act), want)
