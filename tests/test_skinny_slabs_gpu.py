"""Skinny products in K slices (native/kernels/decode_slabs.hip) against the plain product in float64, and the hyper-connection step that adds the slices."""
import pytest
import torch

from kgs.ops import decode as D
from kgs.ops.hyper import hyper_step

pytestmark = pytest.mark.gpu


def _operands(m, n, k, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(m, k + 8, generator=g, device="cuda").bfloat16()[:, :k]  # rows further apart than they are long
    return x, (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).bfloat16()


# the shortest slice (one round of the weights' ring), one chunk more, many; one and two tiles a wave; column tiles full, of one row and short
@pytest.mark.parametrize("n,k", ((64, 128), (64, 256), (1024, 1024), (2048, 2048), (2048, 8192), (192, 384), (4096, 896), (4224, 2048)))
@pytest.mark.parametrize("m", (1, 16, 17, 32, 33, 64))
def test_slices_add_to_the_product(n, k, m):
    x, w = _operands(m, n, k)
    r, ns = D.slab_split(m, n, k)
    got = D.skinny_slabs(x, D.PackedWeight(w))
    assert got.shape == (ns, m, n) and k % (128 * ns) == 0 and n % (64 * r) == 0
    ks = k // ns
    for i in range(ns):
        ref = x[:, i * ks:(i + 1) * ks].double() @ w[:, i * ks:(i + 1) * ks].double().T
        # fp32 sums of ks products of bf16: the roundings of ks additions, on average their root
        assert float((got[i].double() - ref).abs().max()) <= 2.0 ** -24 * ks * float(ref.abs().max())


def test_what_slices_do_not_take():
    for m, n, k in ((0, 2048, 2048), (65, 2048, 2048), (8, 2080, 2048), (8, 2048, 2080)):
        assert D.slab_split(m, n, k) is None
    x, w = _operands(4, 128, 256)
    for pw in (D.PackedWeight(w, swiglu=True), D.PackedWeight(w, fp8=True)):
        with pytest.raises(ValueError):
            D.skinny_slabs(x, pw)


@pytest.mark.parametrize("width", (64, 1023, 1028, 2048, 2052, 4096, 4100))  # both kernels' edges and rows that 16-byte loads cannot read
@pytest.mark.parametrize("parts", (1, 5, 8, 9))
@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float32))
def test_step_adds_parts_as_it_takes_their_sum(dtype, parts, width):
    t, s = 7, 4
    g = torch.Generator(device="cuda").manual_seed(width)
    rnd = lambda *sh: torch.randn(*sh, generator=g, device="cuda")  # noqa: E731
    y = rnd(parts, t, width)
    args = (rnd(s, s), rnd(s), rnd(s), rnd(width))
    total = y[0].clone()
    for p in y[1:]:
        total += p
    a = rnd(t, s, width)
    b = a.clone()
    want = hyper_step(a, total.to(dtype), *args, 1e-5, ld=width + 4)
    got = hyper_step(b, y, *args, 1e-5, dtype=dtype, ld=width + 4)
    assert torch.equal(a, b) and torch.equal(got, want)


@pytest.mark.parametrize("tokens", (1, 256, 257, 512, 513))  # both sides of where a token takes more threads
@pytest.mark.parametrize("width", (1024, 1028, 2048, 3072, 4096))
def test_step_of_few_tokens(width, tokens):
    s = 3
    g = torch.Generator(device="cuda").manual_seed(tokens)
    rnd = lambda *sh: torch.randn(*sh, generator=g, device="cuda")  # noqa: E731
    x, y = rnd(tokens, s, width), rnd(tokens, width).bfloat16()
    mix, out, in_, w = rnd(s, s), rnd(s), rnd(s), rnd(width)
    ref = torch.einsum("tfd,fs->tsd", x.double(), mix.double()) + out.double()[:, None] * y.double()[:, None]
    u = torch.einsum("tsd,s->td", ref, in_.double())
    h = u * torch.rsqrt(u.pow(2).mean(1, keepdim=True) + 1e-5) * w.double()
    got = hyper_step(x, y, mix, out, in_, w, 1e-5)
    assert float((x.double() - ref).abs().max()) < 1e-5 * float(ref.abs().max())  # four products and sums in fp32
    assert bool(((got.double() - h).abs() <= 2.0 ** -8 * h.abs() + 1e-4).all())
