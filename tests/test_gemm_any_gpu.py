"""The GEMM for any size (native/kernels/gemm_any.hip), its K-major form and the linear layer's
backward pass (native/kernels/linear_grad.hip) at the edges of tiles, slices and vectors, against
float64 products of the same bf16 operands."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu
DEV = "cuda"
# bf16 has 8 significant bits: rounding moves a value by up to 2^-8 of its size, so a result by no
# more in the 2-norm (2^-8 / 2.3 on average); fp32 sums of K products add K 2^-24 at most
REL = 2.0 ** -8


def rnd(*shape):
    return (torch.rand(*shape, device=DEV) * 2 - 1).bfloat16()


def rel(got, want):
    return float((got.double() - want).norm() / want.norm())


def run_any(a, b, c, bm, bn, ns, bias=None, epi=0):
    from kgs.ops import _lib

    (M, K), N = a.shape, b.shape[0]
    ws = torch.empty(ns * M * ((N + 7) // 8 * 8), device=DEV)
    rc = _lib.lib().kgs_gemm_bf16_nt_any(a.data_ptr(), b.data_ptr(), c.data_ptr(), None if bias is None else bias.data_ptr(), M, N, K,
                                         a.stride(0), b.stride(0), c.stride(0), epi, bm, bn, ns, ws.data_ptr(), _lib.stream_handle(a.device))
    assert rc == 0, rc


@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (5, 16, 64), (127, 129, 72), (129, 251, 1096), (256, 256, 128), (257, 264, 136), (40, 520, 2056)])
@pytest.mark.parametrize("bm,bn", [(256, 256), (256, 128), (128, 128)])
@pytest.mark.parametrize("ns", [1, 2, 3])
def test_any_tile_and_slices(M, N, K, bm, bn, ns):
    a, b, bias = rnd(M, K), rnd(N, K), torch.randn(N, device=DEV).bfloat16()
    want = a.double() @ b.double().T
    big = torch.full((M + 1, N + 3), 7.0, device=DEV, dtype=torch.bfloat16)  # rows that are not 16-byte aligned
    run_any(a, b, big[:M, :N], bm, bn, ns)
    assert rel(big[:M, :N], want) < REL
    assert bool((big[M] == 7).all()) and bool((big[:, N:] == 7).all())  # nothing written outside
    c = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    run_any(a, b, c, bm, bn, ns, bias, 2)
    assert rel(c, torch.nn.functional.gelu(want + bias.double(), approximate="tanh")) < 2 * REL


MID = [(192, 128), (224, 128), (192, 192), (224, 192), (256, 192), (224, 256)]


@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (225, 200, 72), (193, 385, 136), (448, 264, 1096), (450, 392, 264)])
@pytest.mark.parametrize("bm,bn", MID)
def test_mid_tiles_repeat_the_large_tile_bits(M, N, K, bm, bn):
    """The tiles between plan's three, at their edges: the 256x256 tile's bits, through views whose rows are not 16-byte
    aligned in C and longer than K in A and B; nothing outside is written."""
    A, B = rnd(M + 1, K + 16), rnd(N + 1, K + 8)
    a, b, bias = A[:M, :K], B[1:, :K], torch.randn(N, device=DEV).bfloat16()
    for epi in (0, 2):
        want = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
        run_any(a, b, want, 256, 256, 1, bias, epi)
        big = torch.full((M + 1, N + 3), 7.0, device=DEV, dtype=torch.bfloat16)
        run_any(a, b, big[:M, :N], bm, bn, 1, bias, epi)
        assert torch.equal(big[:M, :N], want)
        assert bool((big[M] == 7).all()) and bool((big[:, N:] == 7).all())
    assert rel(want, torch.nn.functional.gelu(a.double() @ b.double().T + bias.double(), approximate="tanh")) < 2 * REL


# fewer K-tiles than LDS stages, as many, one round of them and one more; 128x128 tiles of one workgroup a CU, also in slices
@pytest.mark.parametrize("K", [8, 64, 72, 128, 192, 200, 256, 264, 320, 448, 520, 1032])
@pytest.mark.parametrize("bm,bn,ns", [(128, 128, 1), (128, 128, 2), (192, 128, 1), (224, 128, 1), (256, 128, 1), (256, 128, 3)])
def test_tiles_of_one_barrier_a_step(bm, bn, ns, K):
    M, N = 2 * bm + 1, 264
    a, b = rnd(M, K), rnd(N, K)
    want, got, large = a.double() @ b.double().T, *(torch.empty(M, N, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    run_any(a, b, got, bm, bn, ns)
    run_any(a, b, large, 256, 256, 1)
    # one rounding to bf16, and the roundings of K fp32 additions
    assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -24 * K * want.abs().max()).all())
    assert ns > 1 or torch.equal(got, large)


@pytest.mark.parametrize("K", [128, 256, 384, 512, 640])
@pytest.mark.parametrize("M", [128, 200])
@pytest.mark.parametrize("bm,bn", [(128, 128), (256, 128), (128, 256)])
def test_w4x_tiles_of_one_barrier_a_step(bm, bn, M, K):
    from kgs.ops.gemm import gemm_nt_w4x, pack_w4x_weight

    a, b = rnd(M, K), rnd(512, K)
    want = gemm_nt_w4x(a, b, bn=256, bm=256)  # two stages
    for w in (b, pack_w4x_weight(b, bn)):
        for nt in (False, True):
            assert torch.equal(gemm_nt_w4x(a, w, bn=bn, bm=bm, nt_weights=nt), want)


# more tiles than CUs, taking turns: two and three rounds, a last one of one tile and of most CUs; one, two and three pairs of K-tiles; off the lines
@pytest.mark.parametrize("M,N,K", [(2049, 8200, 64), (4100, 4104, 128), (3001, 7000, 200), (5000, 8000, 264), (4000, 4200, 1096)])
@pytest.mark.parametrize("bm,bn", [(256, 256), (224, 256), (192, 192)])
def test_tiles_that_take_turns_keep_the_bits(bm, bn, M, N, K):
    a, b, bias = rnd(M, K), rnd(N, K), torch.randn(N, device=DEV).bfloat16()
    got, want = (torch.empty(M, N, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    for epi in (0, 2):
        run_any(a, b, want, 128, 128, 1, bias, epi)  # a workgroup a tile
        for _ in range(2):
            got.fill_(7)
            run_any(a, b, got, bm, bn, 1, bias, epi)
            assert torch.equal(got, want)


def test_tiles_that_take_turns_draw_tickets():
    """A workgroup's tiles behind its first one are tickets of the stream's row of slots: with all of them drawn beforehand each computes that one alone. A
    launch leaves the row cleared, and impossible tickets end its workgroups and are reported."""
    import ctypes

    from kgs.ops import _lib
    from kgs.utils.graph_audit import hip_runtime

    (M, N, K), s, row = (5120, 8192, 192), torch.cuda.Stream(), ctypes.c_void_p()
    a, b, got, want = rnd(M, K), rnd(N, K), torch.zeros(M, N, device=DEV, dtype=torch.bfloat16), torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    run_any(a, b, want, 128, 128, 1)
    _lib.check(_lib.lib().kgs_tile_queue_row(s.cuda_stream, ctypes.byref(row)), "kgs_tile_queue_row")
    torch.cuda.synchronize()
    hip = hip_runtime()
    hip.hipMemcpy.argtypes, hip.hipMemcpy.restype = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int], ctypes.c_int
    tiles, cus = M // 256 * (N // 256), torch.cuda.get_device_properties(DEV).multi_processor_count

    def go(ticket):
        words = (ctypes.c_int * 128)(*([ticket] + [0] * 15) * 8)
        assert hip.hipMemcpy(row, words, 512, 1) == 0  # host to device
        got.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            run_any(a, b, got, 256, 256, 1)
        torch.cuda.synchronize()
        same = (got.view(M // 256, 256, N // 256, 256) == want.view(M // 256, 256, N // 256, 256)).all(dim=3).all(dim=1)
        return int(same.sum()), _lib.tile_queue_check()

    assert go(tiles // 8)[0] == cus < tiles
    done, check = go(0x40000000)
    assert done == cus and check["error_slots"] == 8
    done, check = go(0)
    assert done == tiles and check["dirty_slots"] == check["error_slots"] == 0


# one K-step pair a tile, where a tile's ticket is drawn and handed over within it, and several
@pytest.mark.parametrize("K", [64, 1000])
def test_tiles_that_take_turns_beside_held_cus_and_in_a_graph(K):
    from kgs.ops import _lib
    from kgs.ops.elementwise import cu_hold

    M, N = 4100, 9000
    a, b, want = rnd(M, K), rnd(N, K), torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    run_any(a, b, want, 128, 128, 1)
    side, out = torch.cuda.Stream(), [torch.zeros_like(want) for _ in range(2)]
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        cu_hold(48, 200.0, lds_kb=64)
        run_any(a, b, out[1], 224, 256, 1)  # a slot of its own
    for _ in range(2):
        out[0].zero_()
        run_any(a, b, out[0], 224, 256, 1)
    torch.cuda.synchronize()
    assert all(torch.equal(o, want) for o in out)
    before, g = _lib.tile_queue_stats()["capture_slots"], torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        run_any(a, b, out[0], 224, 256, 1)
    assert _lib.tile_queue_stats()["capture_slots"] == before  # a workgroup a tile
    for _ in range(3):
        out[0].zero_()
        g.replay()
        run_any(a, b, out[1].zero_(), 224, 256, 1)
        torch.cuda.synchronize()
        assert all(torch.equal(o, want) for o in out)
    assert _lib.tile_queue_check()["dirty_slots"] == 0


def tile(M, N, K, gated=False):
    from kgs.ops import _lib

    t = _lib.lib().kgs_gemm_bf16_nt_tile(M, N, K, int(gated))
    return t >> 16, t & 0xffff


# sizes whose tile, by the rule, is each of MID
@pytest.mark.parametrize("M,N,K", [(642, 5480, 128), (965, 5456, 136), (1541, 5008, 128), (1543, 5408, 128), (2035, 4832, 128),
                                   (2054, 5392, 128)])
def test_mid_tiles_with_every_epilogue(M, N, K):
    """What is stored beside the product: the residual sum, both outputs of a training pass."""
    from kgs.ops import gemm_nt
    from kgs.ops.gemm import add_product_, gemm_nt_act

    assert tile(M, N, K) in MID
    a, b, bias = rnd(M, K), rnd(N, K), torch.randn(N, device=DEV).bfloat16()
    z = a.double() @ b.double().T
    assert rel(gemm_nt(a, b), z) < REL
    c0 = rnd(M, N)
    c = c0.clone()
    assert add_product_(a, b, c) and rel(c, z + c0.double()) < 2 * REL
    pre, y = gemm_nt_act(a, b, bias, "silu")
    assert rel(pre, z + bias.double()) < REL
    assert rel(y, torch.nn.functional.silu(pre.double())) < REL


def test_the_sizes_above_have_every_tile():
    assert {tile(*s) for s in ((642, 5480, 128), (965, 5456, 136), (1541, 5008, 128), (1543, 5408, 128), (2035, 4832, 128), (2054, 5392, 128))} == set(MID)


@pytest.mark.parametrize("M,N,K,bm,bn", [(642, 5504, 128, 192, 128), (642, 5456, 136, 192, 128), (965, 5456, 136, 224, 128), (2017, 3184, 328, 224, 128),
                                         (1541, 5120, 128, 224, 256), (1541, 5136, 200, 224, 256), (965, 5504, 128, 128, 128)])
@pytest.mark.parametrize("act", ["silu", "gelu_tanh", "clamped"])
def test_mid_tiles_of_gated_products(M, N, K, bm, bn, act):
    """Each tile, with and without a K tail (which gemm_swiglu itself keeps to the unfused way)."""
    from kgs.ops import _lib
    from kgs.ops.activation import Gate, act_mul
    from kgs.ops.gemm import GATE_ACTS, gemm_swiglu

    assert tile(M, N, K, gated=True) == (bm, bn)
    a, b = rnd(M, K), rnd(N, K)
    both = (a.double() @ b.double().T).bfloat16().double()
    g, u = both.chunk(2, 1)
    gate = Gate("clamped", 1.5) if act == "clamped" else Gate.of(act)
    want = act_mul(both.float(), gate).double() if act == "clamped" else u * (
        torch.nn.functional.silu(g) if act == "silu" else torch.nn.functional.gelu(g, approximate="tanh"))
    got = torch.full((M + 1, N // 2), 7.0, device=DEV, dtype=torch.bfloat16)
    assert _lib.lib().kgs_gemm_bf16_nt_swiglu(a.data_ptr(), b.data_ptr(), got.data_ptr(), M, N, K, K, K, N // 2, GATE_ACTS[gate.act],
                                              gate.limit_ptr(a.device), _lib.stream_handle(a.device)) == 0
    assert rel(got[:M], want) < 2 * REL and bool((got[M] == 7).all())
    if K % 128 == 0 and N % 128 == 0:
        assert torch.equal(gemm_swiglu(a, b, gate), got[:M])


def test_any_reads_nothing_past_its_operands():
    """Views inside larger buffers whose surroundings are NaN: the K tail and the rows past the
    end have to arrive as zeros."""
    from kgs.ops import gemm_nt

    M, N, K = 130, 136, 200
    A, B = (torch.full((r + 2, K + 8), float("nan"), device=DEV, dtype=torch.bfloat16) for r in (M, N))
    a, b = A[1:M + 1, :K], B[1:N + 1, :K]
    a.copy_(rnd(M, K))
    b.copy_(rnd(N, K))
    assert rel(gemm_nt(a, b), a.double() @ b.double().T) < REL


@pytest.mark.parametrize("M,N,K", [(64, 512, 2048), (300, 304, 2400), (128, 640, 4096)])
def test_sliced_products_on_two_streams_and_in_a_graph(M, N, K):
    """Every call has scratch of its own: interleaved products keep their results, and a captured
    one replays to the eager result."""
    from kgs.ops import gemm_nt
    from kgs.ops.gemm import _scratch_floats

    assert _scratch_floats(M, N, K) > 0
    ops = [(rnd(M, K), rnd(N, K)) for _ in range(4)]
    want = [gemm_nt(a, b) for a, b in ops]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    got = []
    for i, (a, b) in enumerate(ops):
        with torch.cuda.stream(streams[i % 2]):
            got.append(gemm_nt(a, b))
    torch.cuda.synchronize()
    assert all(torch.equal(g, w) for g, w in zip(got, want))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = gemm_nt(*ops[0])
    for _ in range(3):
        out.zero_()
        graph.replay()
        gemm_nt(*ops[1])  # eager work between the replays
        torch.cuda.synchronize()
        assert torch.equal(out, want[0])


@pytest.mark.parametrize("M,N,K", [(8, 8, 1), (16, 24, 63), (136, 72, 200), (128, 256, 65), (264, 136, 1096), (64, 512, 2056)])
@pytest.mark.parametrize("ta,tb", [(1, 1), (1, 0), (0, 1)])
@pytest.mark.parametrize("ns", [1, 3])
def test_tr_layouts(M, N, K, ta, tb, ns):
    from kgs.ops import _lib

    if not (ta and tb):
        K = (K + 7) // 8 * 8  # the K-contiguous operand's chunks
    a, b = rnd(K, M) if ta else rnd(M, K), rnd(K, N) if tb else rnd(N, K)
    want = (a.T if ta else a).double() @ (b if tb else b.T).double()
    ws = torch.empty(ns * M * N, device=DEV)
    c = torch.full((M + 1, N), 7.0, device=DEV, dtype=torch.bfloat16)
    rc = _lib.lib().kgs_gemm_bf16_tr(a.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, K, a.stride(0), b.stride(0), N, ta, tb, ns,
                                     ws.data_ptr(), _lib.stream_handle(a.device))
    assert rc == 0
    assert rel(c[:M], want) < REL and bool((c[M] == 7).all())


@pytest.mark.parametrize("act", [None, "gelu", "relu", "silu"])
@pytest.mark.parametrize("M,N", [(1, 8), (7, 3), (64, 64), (65, 136), (513, 72), (1025, 200), (520, 67)])
def test_act_grad(act, M, N):
    """The gradient through an activation, its transpose and its column sums."""
    from kgs.ops.gemm import act_grad

    gy, z = rnd(M, N), 3 * rnd(M, N)
    z[0, 0] = 0.0
    want = gy.double()
    if act:
        x = z.double().requires_grad_(True)
        f = {"gelu": lambda v: torch.nn.functional.gelu(v, approximate="tanh"), "relu": torch.relu, "silu": torch.nn.functional.silu}[act]
        (want,) = torch.autograd.grad(f(x), x, gy.double())
    gz, gzt, gb = act_grad(gy, z, act, True, True)
    assert float((gz.double() - want).abs().max()) < 2 * REL * float(want.abs().max())
    assert torch.equal(gzt, gz.T.contiguous())
    sums = gz.double().sum(0)
    assert float((gb.double() - sums).abs().max()) <= REL * float(sums.abs().max()) + M * 2.0 ** -24 * float(gz.double().abs().sum(0).max())


@pytest.mark.parametrize("act", [None, "gelu", "relu", "silu"])
@pytest.mark.parametrize("rows,din,dout,bias", [(64, 512, 2048, True), (1, 64, 72, True), (100, 136, 200, False), (1001, 264, 128, True),
                                                (33, 7, 10, True), (2048, 256, 512, True)])
def test_linear_training_step(act, rows, din, dout, bias):
    """Output, and the gradients of input, weight and bias, against float64."""
    from kgs.ops import Linear

    lin = Linear(din, dout, bias=bias, act=act, device=DEV)
    if bias:
        with torch.no_grad():
            lin.bias.copy_(torch.randn(dout, device=DEV))
    x, gy = rnd(rows, din).requires_grad_(True), rnd(rows, dout)
    y = lin(x)
    y.backward(gy)
    p = [t.detach().double().requires_grad_(True) for t in [x, lin.weight] + ([lin.bias] if bias else [])]
    z = p[0] @ p[1].T + (p[2] if bias else 0.0)
    f = {None: lambda v: v, "gelu": lambda v: torch.nn.functional.gelu(v, approximate="tanh"), "relu": torch.relu,
         "silu": torch.nn.functional.silu}[act]
    # the kernels' activation and its gradient see z rounded to bf16: up to 2^-8 of z on either side
    want = torch.autograd.grad(f(z), p, gy.double())
    assert rel(y.detach(), f(z).detach()) < 3 * REL
    for got, w in zip([x.grad, lin.weight.grad] + ([lin.bias.grad] if bias else []), want):
        assert rel(got, w) < 8 * REL
    assert y.dtype == torch.bfloat16


def test_linear_keeps_nan_and_skips_what_needs_no_gradient():
    from kgs.ops import Linear

    lin = Linear(64, 64, act="relu", device=DEV)
    x = rnd(8, 64)
    x[3, 5] = float("nan")
    y = lin(x)  # no gradient for x
    assert bool(y[3].isnan().all()) and not bool(y[:3].isnan().any())
    y.backward(torch.ones_like(y))
    assert x.grad is None and lin.weight.grad is not None


@pytest.mark.parametrize("M,N,K", [(1, 256, 128), (130, 512, 384), (257, 1024, 512), (4500, 4096, 384), (8320, 2304, 512),
                                   (512, 512, 2048), (2048, 4096, 512), (2304, 4096, 256)])
def test_products_of_any_rows_add_and_gate_like_their_parts(M, N, K):
    """The residual add and the gated product in the epilogue, on ragged rows of small and of
    persistent grids, against the product and a separate pass."""
    from kgs.ops import gemm_nt
    from kgs.ops.gemm import _scratch_floats, add_product_, gemm_swiglu
    from kgs.ops.transformer import silu_mul

    a, b = rnd(M, K), rnd(N, K)
    c = gemm_nt(a, b)
    assert rel(c, a.double() @ b.double().T) < REL
    x = rnd(M, N)
    want = (x.float() + c.float()).bfloat16()
    assert add_product_(a, b, x)
    assert torch.equal(x, want) if not _scratch_floats(M, N, K) else rel(x, want.double()) < REL
    if N % 128 == 0:
        assert torch.equal(gemm_swiglu(a, b), silu_mul(gemm_nt(a, b, variant="bounded")))


@pytest.mark.parametrize("act", ["gelu_tanh", "clamped"])
@pytest.mark.parametrize("M", [100, 4500])
def test_gated_products_of_any_rows(act, M):
    from kgs.ops.activation import Gate
    from kgs.ops.gemm import gemm_swiglu

    gate = Gate(act, 0.5 if act == "clamped" else 0.0)
    a, w = rnd(M, 512), rnd(4096, 512)
    z = a.double() @ w.double().T
    g, u = z[:, :2048], z[:, 2048:]
    if act == "clamped":
        g, u = g.clamp(max=0.5), u.clamp(-0.5, 0.5)
        want = g * torch.sigmoid(1.702 * g) * (u + 1)
    else:
        want = torch.nn.functional.gelu(g, approximate="tanh") * u
    assert rel(gemm_swiglu(a, w, gate), want) < 3 * REL


@pytest.mark.parametrize("M,N,K", [(256, 256, 768), (256, 768, 1024), (1024, 1024, 4096)])
def test_fp8_small_grids_equal_the_eight_wave_kernel(M, N, K):
    from kgs.ops import gemm_fp8_nt, quantize_fp8

    (a, sa), (b, sb) = quantize_fp8(rnd(M, K)), quantize_fp8(rnd(N, K))
    assert torch.equal(gemm_fp8_nt(a, b, sa, sb), gemm_fp8_nt(a, b, sa, sb, variant="fast"))


@pytest.mark.parametrize("rows,cols,off,rows2,cols2", [(1, 1, 0, 1, 9), (7, 33, 1, 130, 33), (300, 2243, 3, 17, 2243), (64, 4097, 7, 1, 8),
                                                       (513, 64, 1, 2, 5)])
def test_padded_rows(rows, cols, off, rows2, cols2):
    """Copies of rows at any 2-byte alignment, zeros up to the next chunk; even rows come back as they are."""
    from kgs.ops.gemm import _even

    a, b = rnd(rows, cols + off)[:, off:], rnd(rows2, cols2)
    for t, e in zip((a, b), _even(a, b)):
        if t.shape[1] % 8 == 0 and t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0:
            assert e is t
        else:
            assert e.shape[1] % 8 == 0 and torch.equal(e[:, :t.shape[1]], t) and not e[:, t.shape[1]:].any()
    assert torch.equal(_even(a)[0][:, :cols], a)


@pytest.mark.parametrize("M,N,K", [(3, 2, 33), (24, 65, 1555), (128, 130, 2467), (300, 257, 129), (257, 512, 39), (64, 72, 31)])
@pytest.mark.parametrize("act", [None, "gelu"])
def test_odd_rows(M, N, K, act):
    """Rows of no multiple of eight, in every layout, and an aligned K in rows that are not."""
    from kgs.ops import gemm_nt
    from kgs.ops.gemm import gemm_bf16

    a, b, bias = rnd(M, K), rnd(N, K), rnd(1, N)[0]
    want = a.double() @ b.double().T
    y = gemm_nt(a, b, bias=bias if act else None, act=act)
    assert rel(y, torch.nn.functional.gelu(want + bias.double(), approximate="tanh") if act else want) < 2 * REL
    if act:
        return
    for ta, tb in ((0, 1), (1, 0), (1, 1)):
        x, z = (a.T.contiguous() if ta else a), (b.T.contiguous() if tb else b)
        assert rel(gemm_bf16(x, z, trans_a=bool(ta), trans_b=not tb), want) < REL
    w = rnd(M, 72)[:, 3:67]
    v = rnd(N, 64)
    assert rel(gemm_nt(w, v), w.double() @ v.double().T) < REL


@pytest.mark.parametrize("rows,din,dout", [(101, 827, 310), (1024, 310, 54), (56, 2877, 153), (4200, 130, 2049)])
@pytest.mark.parametrize("frozen", [None, "x", "w"])
def test_linear_odd_sizes(rows, din, dout, frozen):
    from kgs.ops import Linear

    lin = Linear(din, dout, act="silu", device=DEV)
    x, gy = rnd(rows, din).requires_grad_(frozen != "x"), rnd(rows, dout)
    lin.weight.requires_grad_(frozen != "w")
    lin(x).backward(gy)
    p = [t.detach().double().requires_grad_(True) for t in (x, lin.weight, lin.bias)]
    want = torch.autograd.grad(torch.nn.functional.silu(p[0] @ p[1].T + p[2]), p, gy.double())
    for t, w in zip((x, lin.weight, lin.bias), want):
        if t.requires_grad:
            assert rel(t.grad, w) < 8 * REL  # as test_linear_training_step


@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (64, 64, 64), (65, 63, 72), (130, 200, 1032), (63, 257, 320), (320, 128, 200)])
@pytest.mark.parametrize("epi", [0, 1, 2, 4])
def test_small_tiles_keep_the_bits(M, N, K, epi):
    """64x64 tiles against 128x128 ones: the same products in the same order, every epilogue, edges of
    tiles, fewer K-tiles than stages; a row below the output stays as it is."""
    a, b, bias = rnd(M, K), rnd(N, K), rnd(1, N)[0].contiguous()
    c1, c2 = (torch.full((M + 1, N), 5.0, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    run_any(a, b, c1[:M], 64, 64, 1, bias if epi else None, epi)
    run_any(a, b, c2[:M], 128, 128, 1, bias if epi else None, epi)
    assert torch.equal(c1, c2) and bool((c1[M] == 5).all())


def test_gelu_over_its_range():
    """The epilogue's gelu and its gradient over every finite bf16 value (and the infinities as before)
    against float64: half a bf16 unit plus a few fp32 units of the exponent's argument."""
    from kgs.ops import gemm_nt
    from kgs.ops.gemm import act_grad

    bits = torch.arange(1 << 16, device=DEV, dtype=torch.int32).to(torch.int16)
    x = bits.view(torch.bfloat16)
    x = x[x.isfinite() & (x.abs() < 1e18)]  # the square stays finite
    x = x[:x.numel() // 8 * 8].view(-1, 1).contiguous()
    one = torch.zeros(8, 8, device=DEV, dtype=torch.bfloat16)
    one[:, 0] = 1
    a = torch.zeros(x.shape[0], 8, device=DEV, dtype=torch.bfloat16)
    a[:, :1] = x
    got = gemm_nt(a, one, act="gelu")[:, 0].double()
    z = x[:, 0].double().requires_grad_(True)
    want = torch.nn.functional.gelu(z, approximate="tanh")
    # below -8 or so the result is under 1e-14 and its relative error is the exponent's: 2 |u| 2^-23
    tol = 2.0 ** -8 * want.abs() * 1.01 + 1e-14
    assert bool(((got - want).abs() <= tol).all())
    (d,) = torch.autograd.grad(want.sum(), z)
    gz, _, _ = act_grad(torch.ones_like(a), a, "gelu", False, False)
    assert bool(((gz[:, 0].double() - d).abs() <= 2.0 ** -8 * d.abs() * 1.01 + 1e-6).all())
    y = gemm_nt(torch.tensor([[float("inf")] + 7 * [0.0]], device=DEV).bfloat16(), one, act="gelu")
    assert bool((y == float("inf")).all())


@pytest.mark.parametrize("M,N,K", [(1, 8, 16), (64, 64, 128), (65, 72, 144), (130, 200, 1040), (256, 256, 1024), (63, 264, 640)])
@pytest.mark.parametrize("epi", [0, 1, 2, 3, 4])
def test_small_fp8_tiles(M, N, K, epi):
    """e4m3 operands on 64x64 tiles at their edges, every epilogue, host and device scales; a row below the
    output stays as it is."""
    from kgs.ops import _lib

    a, b = (rnd(r, K).to(torch.float8_e4m3fn) for r in (M, N))
    bias, scale = rnd(1, N)[0].contiguous(), torch.tensor([0.75], device=DEV)
    z = 0.5 * (a.double() @ b.double().T)
    for ptr in (None, scale.data_ptr()):
        c = torch.full((M + 1, N), 5.0, device=DEV, dtype=torch.bfloat16)
        rc = _lib.lib().kgs_gemm_fp8_nt_dev(a.data_ptr(), b.data_ptr(), c.data_ptr(), bias.data_ptr() if epi else None, M, N, K, K, K, N,
                                            0.5, ptr, epi, 64, _lib.stream_handle(a.device))
        assert rc == 0
        want = z * (0.75 if ptr else 1.0) + (bias.double() if epi else 0.0)
        f = [lambda v: v, lambda v: v, lambda v: torch.nn.functional.gelu(v, approximate="tanh"), torch.relu, torch.nn.functional.silu][epi]
        assert rel(c[:M], f(want)) < 2 * REL and bool((c[M] == 5).all())


@pytest.mark.parametrize("M,N,K", [(24, 88, 128), (1024, 1024, 1024), (512, 512, 4096), (2560, 3200, 576), (2048, 2048, 2048)])
def test_fp8_auto_either_side_of_the_rule(M, N, K):
    from kgs.ops.gemm import gemm_fp8_nt

    a, b = (rnd(r, K).to(torch.float8_e4m3fn) for r in (M, N))
    want = a.double() @ b.double().T
    assert rel(gemm_fp8_nt(a, b), want) < REL and rel(gemm_fp8_nt(a, b, variant="bounded"), want) < REL


@pytest.mark.parametrize("M,N,K", [(1, 64, 130), (70, 100, 129), (300, 304, 2404), (16, 64, 2467), (513, 1030, 257), (64, 64, 65), (4096, 72, 43)])
@pytest.mark.parametrize("odd", ["a", "b", "both"])
@pytest.mark.parametrize("act", [None, "gelu"])
def test_products_through_copies(M, N, K, odd, act):
    """The one call that copies odd operands and multiplies: the bits of the two steps, whichever operand is odd (rows of no
    multiple of 8, or a first value off the 16-byte grid) and with slices."""
    from kgs.ops.gemm import _even, _pads, gemm_nt

    def operand(rows, is_odd):
        k = K if odd == "both" else (K + 7) // 8 * 8
        t = rnd(rows, k + 8)
        return t[:, 3:3 + k] if is_odd and odd != "both" else t[:, :k].contiguous()

    a, b = operand(M, odd != "b"), operand(N, odd != "a")
    bias = rnd(1, N)[0] if act else None
    got, plain = gemm_nt(a, b, bias=bias, act=act), gemm_nt(*_even(a, b), bias=bias, act=act)
    if _pads(M, N, a.shape[1]):
        assert torch.equal(got, plain)
    want = a.double() @ b.double().T
    if act:
        want = torch.nn.functional.gelu(want + bias.double(), approximate="tanh")
    assert rel(got, want) < 2 * REL
    assert rel(plain, want) < 2 * REL


def test_short_odd_rows_are_read_where_they_lie():
    """A copy is a launch and an allocation more: not for short rows of small products."""
    from kgs.ops.gemm import _pads

    assert not _pads(64, 64, 97) and not _pads(1624, 72, 43) and not _pads(4096, 4096, 32) and not _pads(1, 64, 128)
    assert _pads(64, 64, 129) and _pads(1624, 72, 65) and _pads(512, 512, 33) and _pads(4096, 4096, 33)


@pytest.mark.parametrize("M,N,K,short", [(3000, 2801, 64, True), (2901, 2900, 256, True), (3000, 2801, 264, False), (2896, 2896, 64, False), (1000, 2801, 64, False)])
@pytest.mark.parametrize("act", [None, "silu"])
def test_large_odd_outputs_of_short_sums(M, N, K, short, act):
    """Either side of where rows that leave in 2-byte stores go to the element-wise kernel: its bits there."""
    from kgs.ops import gemm_nt

    a, b, bias = rnd(M, K), rnd(N, K), rnd(1, N)[0] if act else None
    got, plain = gemm_nt(a, b, bias=bias, act=act), gemm_nt(a, b, bias=bias, act=act, variant="generic")
    assert torch.equal(got, plain) or not short
    want = a.double() @ b.double().T
    want = torch.nn.functional.silu(want + bias.double()) if act else want
    assert rel(got, want) < 2 * REL and rel(plain, want) < 2 * REL


@pytest.mark.parametrize("M,N,K,off,taken", [(1598, 5680, 4144, 1, True), (2129, 3728, 4616, 1, True), (3567, 15328, 928, 1, False), (1505, 8296, 4336, 1, False),
                                              (3567, 15328, 928, 0, True), (4467, 4608, 7296, 0, True), (2048, 5120, 2048, 0, True), (8192, 8192, 8192, 0, False)])
def test_finer_tiles_where_they_win(M, N, K, off, taken):
    """Rows off the 128-byte lines leave the eight-wave kernel for more than others leave theirs."""
    from kgs.ops import _lib

    assert _lib.lib().kgs_gemm_bf16_nt_finer(M, N, K, 0, off) == taken


@pytest.mark.parametrize("M,N,K,pad,off,taken", [(2560, 3912, 264, 0, 0, True), (2560, 3912, 248, 0, 0, False), (2576, 3584, 712, 0, 0, True), (2576, 3584, 704, 0, 0, False), (2576, 3584, 704, 8, 0, True),
                                                 (2576, 3584, 704, 0, 8, True), (1500, 12344, 3080, 0, 0, True), (259, 264, 264, 0, 0, False)])
@pytest.mark.parametrize("act", [None, "gelu", "silu"])
def test_rows_off_the_lines(M, N, K, pad, off, taken, act):
    """Rows of A that start off the 128-byte lines take the eight-wave kernel where the tiles are as large as its
    own: the same bits as the tiles that any such product can have."""
    from kgs.ops import _lib, gemm_nt
    from kgs.ops.gemm import EPI

    a = torch.full((M + 1, K + pad), float("nan"), device=DEV, dtype=torch.bfloat16).reshape(-1)[off:off + M * (K + pad)].view(M, K + pad)[:, :K]
    b, bias = rnd(N, K), None if act is None else rnd(N)
    a.copy_(rnd(M, K))
    lib = _lib.lib()
    assert lib.kgs_gemm_bf16_nt_off_lines(a.data_ptr(), M, N, K, a.stride(0), 0) == taken
    got, tiles = gemm_nt(a, b, bias=bias, act=act), torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    run_any(a, b, tiles, 256, 256, 1, bias, EPI[act])
    if lib.kgs_gemm_bf16_nt_scratch(M, N, K) == 0:
        assert torch.equal(got, tiles)
    assert rel(got if act is None else gemm_nt(a, b), a.double() @ b.double().T) < REL
