"""Latent attention of a decode step in parts by length, at the lengths where the parts' list can go wrong."""
import numpy as np
import pytest
import torch

from kgs.ops.latent import LatentRows, latent_attention, split_parts, waves_for

pytestmark = pytest.mark.gpu


def lengths(kind, batch):
    rng = np.random.default_rng(batch)
    return {"equal": np.full(batch, 97), "ones": np.ones(batch, int), "one long": np.array([5000] + [1] * (batch - 1)),
            "long last": np.array([33] * (batch - 1) + [4097]), "drawn": rng.integers(1, 900, batch),
            "borders": np.resize([31, 32, 33, 64, 65, 2048, 2049], batch)}[kind]


@pytest.mark.parametrize("kind", ["equal", "ones", "one long", "long last", "drawn", "borders"])
@pytest.mark.parametrize("batch,heads,rp,hr,window", [(3, 16, 512, 64, 0), (24, 16, 512, 0, 0), (65, 5, 128, 32, 0), (128, 16, 384, 0, 100),
                                                      (7, 40, 512, 0, 0), (40, 40, 64, 0, 33), (256, 2, 32, 32, 0)])
def test_parts_by_length(kind, batch, heads, rp, hr, window):
    """Against the softmax in double, and the equal splits; bf16 outputs of sums in fp32: two units of 2^-8 of the largest value,
    the bound of the other latent tests."""
    lens = lengths(kind, batch)
    g = torch.Generator(device="cuda").manual_seed(batch)
    need = -(-lens // 32)
    W = int(need.max()) + 1
    ids = 1 + np.random.default_rng(1).permutation(int(need.sum()))
    bt = np.zeros((batch, W), np.int32)
    at = 0
    for b, c in enumerate(need):
        bt[b, :c] = ids[at:at + c]
        at += c
    pages = torch.randn(len(ids) + 1, 32, rp + hr, device="cuda", generator=g).bfloat16()
    q = torch.randn(batch, heads * (rp + hr), device="cuda", generator=g).bfloat16()
    i32 = dict(dtype=torch.int32, device="cuda")
    pos, ar = torch.tensor(lens - 1, **i32), torch.arange(batch, **i32)
    waves = waves_for(heads, rp)
    tiles = -(-heads // (16 * waves))
    parts = split_parts(batch, tiles, max(W, 4), rp)
    assert parts > batch
    rows = dict(nt=batch, q0=ar, n=torch.ones(batch, **i32), pos0=pos, bt=torch.tensor(bt, **i32), tok_seq=ar, tok_pos=pos, rows=None,
                items=None, ntiles=batch * tiles, tiles=tiles, waves=waves, nsplit=1)
    scale = (rp + hr) ** -0.5
    got = latent_attention(q, pages, LatentRows(**rows, parts=parts), heads, scale, hr, window).float()
    want = torch.empty(batch, heads, rp, dtype=torch.float64, device="cuda")
    for b, n in enumerate(lens):
        lo = max(0, n - window) if window else 0
        c = pages[torch.tensor(bt[b, :need[b]], device="cuda").long()].reshape(-1, rp + hr)[lo:n].double()
        want[b] = torch.softmax(q[b].view(heads, -1).double() @ c.T * scale, -1) @ c[:, :rp]
    bound = 2 * 2.0 ** -8 * want.abs().max().item()
    assert (got.view(batch, heads, rp) - want).abs().max().item() < bound
    whole = latent_attention(q, pages, LatentRows(**rows), heads, scale, hr, window).float()
    assert (got - whole).abs().max().item() < bound


@pytest.mark.parametrize("lens,parts,pages", [([79] * 8, 256, 1), ([500, 33, 1, 32], 256, 1), ([5000] + [1] * 7, 256, 3), ([2000] * 24, 256, 7)])
def test_parts_are_as_short_as_the_places_allow(lens, parts, pages):
    """A page each where there are places for all, else as few as make them fit (64 parts of a sequence at most)."""
    from kgs.ops import _lib

    nt, heads, rp = len(lens), 16, 128
    i32 = dict(dtype=torch.int32, device="cuda")
    W = -(-max(lens) // 32)
    ar, pos, bt = torch.arange(nt, **i32), torch.tensor(lens, **i32) - 1, torch.zeros(nt, W, **i32)
    cache, q = (torch.randn(*s, device="cuda").bfloat16() for s in ((1, 32, rp), (nt, heads * rp)))
    o, po, ml, of = torch.empty_like(q), torch.empty(parts, heads, rp, device="cuda"), torch.empty(parts, heads, 2, device="cuda"), torch.full((nt, 2), -1, **i32)
    one = torch.ones(nt, **i32)
    assert _lib.lib().kgs_latent_attn_parts(q.data_ptr(), cache.data_ptr(), o.data_ptr(), po.data_ptr(), ml.data_ptr(), of.data_ptr(), ar.data_ptr(),
                                            one.data_ptr(), pos.data_ptr(), bt.data_ptr(), 1, 1, parts, heads, W, nt, rp, 0, 0, 0.1,
                                            _lib.stream_handle(q.device)) == 0
    want = [-(-(-(-n // 32)) // pages) for n in lens]
    assert of[:, 1].tolist() == want and of[:, 0].tolist() == [sum(want[:i]) for i in range(nt)]
