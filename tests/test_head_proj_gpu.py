"""Per-head projections of few tokens, at the edges of their tiles of tokens and of the loads that are in flight together."""
import pytest
import torch

from kgs.ops.latent import head_proj

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [32, 128, 480, 512, 544, 1024])
@pytest.mark.parametrize("nt,H,N", [(1, 16, 128), (16, 3, 16), (17, 16, 512), (32, 2, 48), (33, 32, 128), (64, 5, 128), (130, 1, 64),
                                    (65, 64, 128)])
@pytest.mark.parametrize("each", [None, False, True])
def test_few_tokens(nt, H, N, K, each):
    """bf16 outputs of fp32 sums: 2^-8 of the largest value covers the rounding (2^-9) and the sigmoid's and the sums' errors."""
    g = torch.Generator(device="cuda").manual_seed(nt + K)
    a = torch.randn(nt, H * K, device="cuda", generator=g).bfloat16()
    w = (torch.randn(H, N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    gate = None if each is None else torch.randn(nt + 2, H * N if each else H, device="cuda", generator=g).bfloat16()
    rows = torch.randperm(nt + 2, device="cuda", generator=g)[:nt].int()
    out = torch.full((nt + 2, H * N), 7.0, device="cuda", dtype=torch.bfloat16)
    head_proj(a, w, nt, out, rows_out=rows, gate=gate, each=bool(each))
    want = torch.full((nt + 2, H, N), 7.0, device="cuda", dtype=torch.float64)
    y = (w.double() @ a.double().view(nt, H, K, 1)).squeeze(-1)
    if gate is not None:
        y *= torch.sigmoid(gate.double().view(nt + 2, H, -1))[rows.long()]
    want[rows.long()] = y
    got = out.double().view(nt + 2, H, N)
    assert (got - want).abs().max() < 2.0 ** -8 * y.abs().max()
    rest = torch.ones(nt + 2, dtype=torch.bool, device="cuda")
    rest[rows.long()] = False
    assert torch.equal(got[rest], want[rest])
