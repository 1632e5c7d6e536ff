"""The native autograd node of ``kgs.ops.Linear`` against the Python function that runs the same kernels
(itself held to float64 in test_gemm_any_gpu.py): the same bits, and the same answers where only
Python's can run."""
import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("own_rng")]
DEV = "cuda"


def rnd(*s):
    return torch.randn(*s, device=DEV).bfloat16()


def leaves(rows, din, dout, bias):
    return [t.requires_grad_(True) for t in (rnd(rows, din), rnd(dout, din) * din ** -0.5)] + [rnd(dout).requires_grad_(True) if bias else None]


# edges: one row, sums of one chunk, odd columns of either side (padded copies), rows of no multiple of 8, K slices
SHAPES = [(1, 64, 72), (64, 512, 2048), (100, 136, 200), (1001, 264, 128), (33, 131, 74), (7, 520, 131), (129, 8, 8)]


@pytest.mark.parametrize("act", [None, "gelu", "relu", "silu"])
@pytest.mark.parametrize("rows,din,dout", SHAPES)
@pytest.mark.parametrize("bias", [True, False])
def test_same_bits(act, rows, din, dout, bias):
    from kgs.ops.gemm import _LinearFn, linear

    x, w, b = leaves(rows, din, dout, bias)
    gy, ins = rnd(rows, dout), [t for t in (x, w, b) if t is not None]
    y, ref = linear(x, w, b, act), _LinearFn.apply(x, w, b, act)
    assert "LinearNode" in y.grad_fn.name() and "LinearNode" not in ref.grad_fn.name()
    assert torch.equal(y, ref)
    want = torch.autograd.grad(ref, ins, gy, retain_graph=True)
    for got, t in zip(torch.autograd.grad(y, ins, gy, retain_graph=True), want):
        assert torch.equal(got, t)
    for i, t in enumerate(ins):  # one of the gradients, and of a gradient that is no contiguous matrix
        (got,) = torch.autograd.grad(y, t, gy.T.contiguous().T, retain_graph=True)
        assert torch.equal(got, want[i])
    with torch.no_grad():
        assert torch.equal(linear(x, w, b, act), ref)
        assert torch.equal(linear(x.detach(), w.detach(), None if b is None else b.detach(), act),
                           _LinearFn.apply(x.detach(), w.detach(), None if b is None else b.detach(), act))


def test_without_the_node(monkeypatch):
    from kgs.ops import _lib
    from kgs.ops.gemm import linear

    x, w, b = leaves(64, 512, 256, True)
    gy = rnd(64, 256)
    want = linear(x, w, b, "gelu")
    monkeypatch.setattr(_lib, "autograd", lambda: None)
    got = linear(x, w, b, "gelu")
    assert "_LinearFn" in got.grad_fn.name() and torch.equal(got, want)
    for g, t in zip(torch.autograd.grad(got, (x, w, b), gy), torch.autograd.grad(want, (x, w, b), gy)):
        assert torch.equal(g, t)


def test_rows_apart_and_large_products_keep_their_ways():
    from kgs.ops.gemm import _LinearFn, linear

    x, w, b = leaves(64, 256, 128, True)
    wide = rnd(64, 300)[:, 3:259].requires_grad_(True)  # rows of 300, off the 16-byte chunks
    assert torch.equal(linear(wide, w, b, "gelu"), _LinearFn.apply(wide, w, b, "gelu"))
    x, w, b = leaves(4096, 4096, 4096, False)
    assert "LinearNode" not in linear(x, w).grad_fn.name()
    x, w, b = leaves(64, 20, 24, False)  # short odd rows: element by element
    assert torch.equal(linear(x, w), _LinearFn.apply(x, w, None, None))


def test_saved_tensor_hooks_see_every_saved_matrix():
    from kgs.ops.gemm import linear

    x, w, b = leaves(64, 128, 256, True)
    gy = rnd(64, 256)
    want = torch.autograd.grad(linear(x, w, b, "gelu"), (x, w, b), gy)
    with torch.autograd.graph.save_on_cpu():
        y = linear(x, w, b, "gelu")
    assert all(torch.equal(a, c) for a, c in zip(torch.autograd.grad(y, (x, w, b), gy), want))
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t.cpu()):
        y = linear(x, w, b, "gelu")
    with pytest.raises(RuntimeError, match="saved tensor"):
        torch.autograd.grad(y, (x, w, b), gy)
    y = linear(x, w, b, "gelu")
    with torch.no_grad():
        w.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(y, (x, w, b), gy)


def test_python_only_calls_keep_their_answers():
    """Transforms and tangents are refused as by the Python function; a trace records a call of it."""
    import torch.autograd.forward_ad as fwd

    from kgs.ops.gemm import _LinearFn, linear

    x, w, b = leaves(64, 128, 256, True)

    def refusal(f):
        try:
            f()
        except Exception as e:  # noqa: BLE001 -- its type and text are compared
            return type(e), str(e)
        return None

    def tangent(f):
        with fwd.dual_level():
            f(fwd.make_dual(x.detach(), torch.ones_like(x)), w.detach(), b.detach(), "gelu")

    def under_vmap(f):
        torch.vmap(lambda v: f(v, w, b, "gelu"))(x.detach().reshape(4, 16, 128))

    for how in (tangent, under_vmap, lambda f: f(x.detach().cpu(), w.detach().cpu(), None, None), lambda f: f(x, w[:, :64], b, None),
                lambda f: f(x.float(), w, b, None), lambda f: f(x, w, b[:8], "gelu"), lambda f: f(x, w, b, "tanh")):
        assert refusal(lambda: how(linear)) == refusal(lambda: how(_LinearFn.apply))
        assert refusal(lambda: how(linear)) is not None
    assert "LinearNode" in linear(x, w, b, "gelu").grad_fn.name()  # nothing stays behind of the refused ones
    graph = torch.jit.trace(lambda *v: linear(*v, "gelu"), tuple(t.detach() for t in (x, w, b)), check_trace=False).graph
    assert "_LinearFn" in str(graph)


def test_transforms_leave_nothing_behind():
    """Inside a transform the Python function, which has no rule for one; after it the node again."""
    from kgs.ops.gemm import linear

    x, w, b = leaves(64, 128, 256, True)
    one = torch.ones(3, device=DEV)
    for transform in (lambda f: torch.vmap(f)(one), lambda f: torch.func.grad(lambda v: f(v).sum())(one), lambda f: torch.func.jvp(f, (one,), (one,))):
        transform(lambda v: v * 2)
        assert "LinearNode" in linear(x, w, b, "gelu").grad_fn.name()
        with pytest.raises(RuntimeError, match="setup_context"):
            transform(lambda v: linear(x, w, b, "gelu").sum() * v)
        assert "LinearNode" in linear(x, w, b, "gelu").grad_fn.name()


def test_backward_of_streams_threads_and_graphs():
    import threading

    from kgs.ops.gemm import linear

    def step(x, w, b, gy):
        y = linear(linear(x, w, b, "gelu"), w, b, "silu")
        assert "LinearNode" in y.grad_fn.name()
        return torch.autograd.grad(y, (x, w, b), gy)

    sets = [(*leaves(96, 256, 256, True), rnd(96, 256)) for _ in range(4)]
    want = [step(*s) for s in sets]
    got = [None] * 4

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(8):
                got[i] = step(*sets[i])
            torch.cuda.current_stream().synchronize()

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    for a, c in zip(got, want):
        assert all(torch.equal(g, h) for g, h in zip(a, c))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step(*sets[0])
    for _ in range(3):
        [t.zero_() for t in out]
        graph.replay()
        assert all(torch.equal(g, h) for g, h in zip(out, want[0]))
        torch.cuda.synchronize()
