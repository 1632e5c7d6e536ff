"""The gate kernel of few rows (gemm_gate in native/kernels/gemm_any.hip): edges of its tiles, halves and K-steps against float64, the
same bits as the larger tiles', its rule's bounds."""
import pytest
import torch

from kgs.ops import decode as D

pytestmark = pytest.mark.usefixtures("own_rng")
DEV = "cuda"
REL = 2.0 ** -8


def rnd(*s, scale=1.0):
    return (scale * torch.randn(*s, device=DEV)).bfloat16()


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["silu", "gelu_tanh", "clamped"])
@pytest.mark.parametrize("M,I,K", [(1, 8, 8), (63, 24, 72), (64, 32, 64), (65, 40, 136), (127, 520, 200), (128, 1000, 264), (129, 33 * 8, 520),
                                   (200, 96, 2048)])
@pytest.mark.parametrize("bm", [64, 128])
def test_against_float64(M, I, K, act, bm):
    from kgs.ops.activation import Gate
    from kgs.ops.gemm import gemm_gate

    gate = Gate.of(act) if act != "clamped" else Gate("clamped", 1.5)
    a, w = rnd(M, K + 16)[:, 8:8 + K], rnd(2 * I, K + 8, scale=K ** -0.5)[:, :K]
    out = torch.full((M + 1, I + 8), 7.0, device=DEV).bfloat16()
    gemm_gate(a, w, bm, gate, out=out[:M, :I])
    g, u = (a.double() @ w[:I].double().T), (a.double() @ w[I:].double().T)
    if act == "silu":
        want = torch.nn.functional.silu(g) * u
    elif act == "gelu_tanh":
        want = torch.nn.functional.gelu(g, approximate="tanh") * u
    else:
        from kgs.ops.activation import act_mul

        want = act_mul(torch.cat([g, u], 1).float(), gate).double()
    got = out[:M, :I].double()
    # gate, up and their product are rounded to bf16: up to 2^-9 of each, the gate's slope below 1.2 (clamped: 2)
    assert float((got - want).norm() / want.norm()) < 2 * REL
    assert bool((out[M] == 7).all()) and bool((out[:, I:] == 7).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(33, 4096, 1024), (64, 16384, 2048), (65, 8192, 2048), (100, 16384, 2048), (128, 12288, 256)])
def test_same_bits_as_the_larger_tiles(M, N, K):
    from kgs.ops.gemm import gemm_gate, gemm_swiglu

    a, w = rnd(M, K), rnd(N, K, scale=K ** -0.5)
    for bm in (64, 128):
        assert torch.equal(gemm_gate(a, w, bm), gemm_swiglu(a, w))


@pytest.mark.gpu
def test_what_it_refuses():
    from kgs.ops._lib import KernelError
    from kgs.ops.gemm import gemm_gate

    a, w = rnd(8, 64), rnd(32, 64)
    for bad in (lambda: gemm_gate(a, w, 96), lambda: gemm_gate(rnd(8, 65)[:, 1:], w, 64), lambda: gemm_gate(a, rnd(24, 64), 64),
                lambda: gemm_gate(rnd(8, 60), rnd(32, 60), 64), lambda: gemm_gate(a, w, 64, out=rnd(8, 20)[:, :16])):
        with pytest.raises(KernelError):
            bad()
    for bad in (lambda: gemm_gate(a, rnd(32, 72), 64), lambda: gemm_gate(a, w, 64, out=rnd(8, 24))):
        with pytest.raises(ValueError):
            bad()


def test_rule_stays_in_its_bounds():
    for m in (0, 1, 33, 64, 65, 128, 129):
        for n in (16, 24, 4096, 8192, 8208, 16384, 16400, 28672, 28688):
            for k in (8, 12, 2048, 2056, 4096, 8192):
                free, sliced = D.gate_rule(m, n, k, False), D.gate_rule(m, n, k, True)
                assert free in (None, 64, 128) and sliced in (None, free)
                assert free is None or (0 < m <= 128 and n % 16 == 0 and k % 8 == 0 and n <= (28672 if m <= 64 else 16384))
                assert free != 128 or (m > 64 and n > 8192)
