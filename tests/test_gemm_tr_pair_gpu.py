"""A linear layer's two gradient products in one launch: the bits of two launches (themselves held to float64 in
test_gemm_any_gpu.py), in K slices on either side."""
import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("own_rng")]


def rnd(*s):
    return torch.randn(*s, device="cuda").bfloat16()


# m, n, k, slices of dX and dW: one tile each, remainders of rows, columns and sums, odd columns out, more slices than chunks of 128,
# more tiles than one launch takes
@pytest.mark.parametrize("m,n,k,nsx,nsw", [(128, 128, 128, 1, 1), (1, 8, 8, 1, 1), (130, 520, 264, 1, 1), (64, 2048, 512, 4, 1),
                                           (1001, 136, 392, 1, 3), (600, 1000, 129, 2, 4), (257, 384, 515, 64, 64), (2056, 4096, 4104, 1, 1)])
def test_bits_of_two_launches(m, n, k, nsx, nsw):
    from kgs.ops import _lib

    so, stream = _lib.lib(), torch.cuda.current_stream().cuda_stream
    k8 = (k + 7) // 8 * 8
    dy, w, x = rnd(m, n), rnd(n, k8)[:, :k], rnd(m, k8)[:, :k]
    wsx, wsw = (torch.empty(ns * r * k8, device="cuda") for ns, r in ((nsx, m), (nsw, n)))
    want = [torch.empty(r, k, device="cuda", dtype=torch.bfloat16) for r in (m, n)]
    got = [torch.full_like(t, float("nan")) for t in want]
    for a, b, c, r, s, ta, ns, ws in ((dy, w, want[0], m, n, 0, nsx, wsx), (dy, x, want[1], n, m, 1, nsw, wsw)):
        assert so.kgs_gemm_bf16_tr(a.data_ptr(), b.data_ptr(), c.data_ptr(), r, k, s, n, k8, k, ta, 1, ns, ws.data_ptr(), stream) == 0
    rc = so.kgs_gemm_bf16_tr_pair(dy.data_ptr(), w.data_ptr(), x.data_ptr(), *(t.data_ptr() for t in got), m, n, k, n, k8, k8, nsx, nsw,
                                  wsx.data_ptr(), wsw.data_ptr(), stream)
    assert rc == 0
    for a, b in zip(got, want):
        assert torch.equal(a, b)
