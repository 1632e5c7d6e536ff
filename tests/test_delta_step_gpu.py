"""Decoded tokens of the delta rule in one launch: the bits of the three launches that portions take (held to float64 in
test_hybrid_ops_gpu.py), of outputs, states and convolution tails; slot 0 left alone."""
import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("own_rng")]


# heads, rows a sequence (as many in all as sequences), first positions, slots
@pytest.mark.parametrize("H,n,pos,slot", [(1, [1], [0], [1]), (3, [1, 1, 1], [7, 0, 1], [2, 3, 1]), (16, [1] * 5, [9, 4, 0, 0, 3], [4, 0, 2, 0, 5]),
                                          (2, [3, 0, 2, 0, 0], [5, 8, 0, 0, 2], [3, 1, 2, 4, 0])])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("extra", [0, 34])
def test_bits_of_three_launches(H, n, pos, slot, dtype, extra):
    from kgs.ops.delta import DeltaShape, DeltaState, RaggedSeqs, delta_forward, delta_out, delta_step, step_takes

    sh, B, hk = DeltaShape(H, H, 128, 128, 4), len(n), H * 128
    z = torch.randn(B, 3 * hk + 2 * H + 6 + extra, device="cuda").to(dtype)
    offs = (2, 2 + hk, 4 + 2 * hk, 4 + 3 * hk + 1)
    a2, gate = (torch.randn(B, hk + extra, device="cuda").to(dtype) for _ in range(2))
    par = torch.randn(4, 3 * hk, device="cuda"), torch.rand(H, device="cuda"), torch.randn(hk, device="cuda")
    w, ld = torch.randn(128, device="cuda"), hk + extra
    states = [DeltaState(sh, 6, "cuda") for _ in range(2)]
    for t, u in zip(vars(states[0]).values(), vars(states[1]).values()):
        u.copy_(t.normal_())
    start = states[1].S[0].clone(), states[1].conv[0].clone()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    first = [sum(n[:i]) for i in range(B)]
    seqs = RaggedSeqs(i32([b for b in range(B) for _ in range(n[b])]), i32(first), i32(n), i32(pos), i32(slot))
    assert step_takes(z, offs, a2, gate, sh, seqs, ld)
    want = delta_out(delta_forward(z, offs, a2, *par, sh, states[0], seqs), w, gate, 1e-5, ld)
    got = delta_step(z, offs, a2, *par, sh, states[1], seqs, w, gate, 1e-5, ld)
    for b in range(B):
        if slot[b] == 0:
            want[first[b]:first[b] + n[b]] = 0
    assert torch.equal(got, want)
    assert torch.equal(states[1].S[1:], states[0].S[1:]) and torch.equal(states[1].conv[1:], states[0].conv[1:])
    assert torch.equal(states[1].S[0], start[0]) and torch.equal(states[1].conv[0], start[1])


def test_what_it_does_not_take():
    from kgs.ops.delta import DeltaShape, DeltaState, RaggedSeqs, delta_step, step_takes

    z = torch.zeros(2, 400, device="cuda")
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    one, two = RaggedSeqs(i32(0, 0), i32(0), i32(2), i32(0), i32(1)), RaggedSeqs(i32(0, 1), i32(0, 1), i32(1, 1), i32(0, 0), i32(1, 2))
    sh, offs = DeltaShape(1, 1, 128, 128, 4), (0, 128, 256, 384)
    a2 = torch.zeros(2, 128, device="cuda")
    assert step_takes(z, offs, a2, a2, sh, two, 128)
    assert not step_takes(z, offs, a2, a2, sh, one, 128)  # two rows of one sequence
    assert not step_takes(z, offs, a2, a2, sh, two, 129) and not step_takes(z, (1, 129, 257, 385), a2, a2, sh, two, 128)
    for other in (DeltaShape(2, 1, 128, 128, 4), DeltaShape(1, 1, 64, 128, 4), DeltaShape(1, 1, 128, 100, 4), DeltaShape(1, 1, 128, 128, 3)):
        assert not step_takes(z, offs, a2, a2, other, two, 256)
    with pytest.raises(ValueError):
        delta_step(z, offs, a2, torch.zeros(4, 384, device="cuda"), torch.zeros(1, device="cuda"), torch.zeros(128, device="cuda"), sh,
                   DeltaState(sh, 2, "cuda"), one, torch.ones(128, device="cuda"), a2, 1e-5, 128)
