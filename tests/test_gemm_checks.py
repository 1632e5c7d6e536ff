"""What gemm_bf16 refuses before anything is launched, in each of the four layouts, and which kernel a
residual product asks for (no GPU: tensors that only claim to be on one, and a kernel library that
must not be reached, or that only says what was called)."""
import pytest
import torch

from kgs.ops import _lib
from kgs.ops import gemm as G


class Claimed(torch.Tensor):
    """A CPU tensor that says it is on a GPU."""
    is_cuda = True
    gpu = 0

    @property
    def device(self):
        return torch.device("cuda", self.gpu)


def claimed(*shape, dtype=torch.bfloat16, gpu=0):
    t = torch.zeros(*shape, dtype=dtype).as_subclass(Claimed)
    t.gpu = gpu
    return t


class Reached(Exception):
    pass


@pytest.fixture(autouse=True)
def no_library(monkeypatch):
    def lib():
        raise Reached

    monkeypatch.setattr(_lib, "lib", lib)
    for f in (G._tr_slices, G._scratch_floats):
        f.cache_clear()


M, N, K = 64, 72, 128
LAYOUTS = [(ta, tb) for ta in (False, True) for tb in (False, True)]


def operands(ta, tb, n=N):
    return claimed(*((K, M) if ta else (M, K))), claimed(*((n, K) if tb else (K, n)))


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("n", [N, 256])
@pytest.mark.parametrize("bad", ["float32", "uint8", "strided", "cpu", "shape", "device", "vector"])
def test_out_is_checked(ta, tb, n, bad):
    a, b = operands(ta, tb, n)
    out = {"float32": lambda: claimed(M, n, dtype=torch.float32), "uint8": lambda: claimed(M, n, dtype=torch.uint8),
           "strided": lambda: torch.zeros(M, 2 * n, dtype=torch.bfloat16).as_subclass(Claimed)[:, ::2],
           "cpu": lambda: torch.zeros(M, n, dtype=torch.bfloat16), "shape": lambda: claimed(M, n - 8),
           "device": lambda: claimed(M, n, gpu=1), "vector": lambda: claimed(M * n)}[bad]()
    with pytest.raises(TypeError if bad in ("float32", "uint8") else ValueError):
        G.gemm_bf16(a, b, trans_a=ta, trans_b=tb, out=out)


@pytest.mark.parametrize("ta,tb", LAYOUTS)
def test_operands_share_a_device(ta, tb):
    a, b = operands(ta, tb)
    b.gpu = 1
    with pytest.raises(ValueError, match="different devices"):
        G.gemm_bf16(a, b, trans_a=ta, trans_b=tb)


@pytest.mark.parametrize("ta,tb", LAYOUTS)
def test_a_good_out_goes_on(ta, tb):
    a, b = operands(ta, tb)
    with pytest.raises(Reached):
        G.gemm_bf16(a, b, trans_a=ta, trans_b=tb, out=claimed(M, N))


@pytest.mark.parametrize("m,n,entry", [(512, 4096, "kgs_gemm_bf16_nt_add"), (2048, 4096, "kgs_gemm_bf16_nt_add"), (2304, 4096, "kgs_gemm_bf16_nt_addc"),
                                       (4000, 4096, "kgs_gemm_bf16_nt_add"), (8192, 4096, "kgs_gemm_bf16_nt_addc")])
def test_residual_products_of_few_tiles_do_not_take_the_largest_ones(m, n, entry, monkeypatch):
    """256x256 tiles on fewer than half the CUs take up to three times as long as smaller tiles and slices."""
    called = []

    class Library:
        def __getattr__(self, name):
            def call(*args):
                called.append(name)
                return int(name == "kgs_gemm_bf16_nt_w4_ok" and args[3] % 256 == 0)

            return call

    monkeypatch.setattr(_lib, "lib", Library)
    monkeypatch.setattr(_lib, "stream_handle", lambda device=None: 0)
    monkeypatch.delenv("KGS_PREFILL_ADDC", raising=False)
    assert G.add_product_(claimed(m, 128), claimed(n, 128), claimed(m, n))
    assert called[-1] == entry and not ("nt_addc" in entry) ^ ("kgs_gemm_bf16_nt_addc" in called)
