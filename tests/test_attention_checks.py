"""What attention_blocks refuses before anything is launched (no GPU: tensors that only claim to be on
one, and a kernel library that must not be reached)."""
import pytest
import torch

from kgs.ops import _lib
from kgs.ops import transformer as T

H, KV, ROWS = 4, 2, 5


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
    monkeypatch.setattr(torch, "empty", lambda *a, **kw: None)


def call(**other):
    a = dict(q=claimed(ROWS, 128 * H), k=claimed(ROWS, 128 * KV), v=claimed(ROWS, 128 * KV), items=claimed(1, 4, dtype=torch.int32),
             out=claimed(ROWS, 128 * H), k2=claimed(ROWS, 128 * KV), v2=claimed(ROWS, 128 * KV),
             merges=claimed(1, 4, dtype=torch.int32), slots=2)
    a.update(other)
    T.attention_blocks(a.pop("q"), a.pop("k"), a.pop("v"), a.pop("items"), H, KV, a.pop("out"), **a)


@pytest.mark.parametrize("other", [{}, {"k2": None, "v2": None}, {"merges": None, "slots": 0}, {"q": claimed(ROWS, 1024)}])
def test_what_fits_is_launched(other):
    with pytest.raises(Reached):
        call(**other)


@pytest.mark.parametrize("name", ["q", "k", "v", "k2", "v2", "out"])
@pytest.mark.parametrize("bad", [torch.zeros(ROWS, 512, dtype=torch.bfloat16), claimed(ROWS, 512, dtype=torch.float16), claimed(ROWS, 128)])
def test_operands(name, bad):
    with pytest.raises((TypeError, ValueError)):
        call(**{name: bad})


@pytest.mark.parametrize("other", [{"items": torch.zeros(1, 4, dtype=torch.int32)}, {"merges": torch.zeros(1, 4, dtype=torch.int32)},
                                   {"items": claimed(1, 4, dtype=torch.int32, gpu=1)}, {"k2": None}, {"slots": 1},
                                   {"k2": claimed(ROWS, 256, gpu=1)}, {"out": claimed(ROWS - 1, 512)}, {"v": claimed(ROWS - 1, 256)}])
def test_plans_and_places(other):
    with pytest.raises(ValueError):
        call(**other)
