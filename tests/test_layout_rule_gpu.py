"""Products with a K-major right operand by either of their ways (turn_b in native/kernels/gemm_any.hip): the rule's two sides, and
what gemm_bf16 makes of both against float64."""
import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("own_rng")]


def test_prices_the_tiles_that_run():
    """Aligned products of more tiles than CUs run on 256x256 ones, whatever finer tile would fill the CUs better."""
    from kgs.ops.gemm import _tr_slices, _turn_b

    assert not any(_turn_b(*s) for s in ((3072, 6656, 1536), (2304, 8192, 6912), (3584, 9984, 1024), (3840, 8960, 7168), (3584, 5120, 1792)))
    assert _tr_slices(1280, 5376, 11776, False, True) and not _tr_slices(4608, 2560, 512, False, True)


def test_transposes_where_the_reading_kernel_leaves_cus_idle():
    from kgs.ops.gemm import _turn_b

    assert all(_turn_b(*s) for s in ((2048, 1024, 4096), (4096, 512, 4096), (4096, 2048, 8192), (256, 256, 8192)))
    assert not any(_turn_b(*s) for s in ((4096, 8192, 2048), (2048, 14336, 4096), (8192, 2048, 2048), (8192, 14336, 4096)))


@pytest.mark.parametrize("M,N,K", [(2048, 1024, 1024), (4096, 512, 4096), (1024, 4096, 2048), (4352, 1024, 2048), (256, 256, 128)])
@pytest.mark.parametrize("ta", [False, True])
def test_either_way(monkeypatch, M, N, K, ta):
    from kgs.ops import gemm as G

    a = torch.randn(*((K, M) if ta else (M, K)), device="cuda").bfloat16()
    b = torch.randn(K, N, device="cuda").bfloat16()
    want = (a.T if ta else a).double() @ b.double()
    for turn in (None, True, False):
        if turn is not None:
            monkeypatch.setattr(G, "_tr_slices", lambda *s: 0)
            monkeypatch.setattr(G, "_turn_b", lambda *s: turn)
        got = G.gemm_bf16(a, b, trans_a=ta).double()
        assert float((got - want).norm() / want.norm()) < 2.0 ** -8  # one rounding to bf16
