"""What the rules of layers in slices (kgs/serve/model.py) cost a prompt step, whose launches the host gives one by one."""
import types

import pytest

from kgs.ops import decode as D
from kgs.serve.model import ServingModel


class _Untouched:
    def __getitem__(self, i):
        raise AssertionError("the weights were looked at")


def _model(packed):
    m = object.__new__(ServingModel)
    m.cfg, m.packed, m.backend, m.decode_fp8, m.fuse_splitk, m.rope_attn, m.fused_max_batch = types.SimpleNamespace(hidden=4096), packed, "kgs", False, True, False, 64
    return m


@pytest.mark.parametrize("rows", (1, 32, 129, 512, 8192))
def test_rows_outside_are_turned_away_at_once(rows):
    m = _model(_Untouched())
    assert not m._slab_prompts(rows) and not m._wide(rows) and not m._slabs_pay(rows)


def test_each_range_asks_its_own_rule():
    def w(n, k, rope=None):
        return types.SimpleNamespace(n=n, k=k, rope=rope)

    m = _model([{"qkv": w(6144, 4096, (32, 8)), "o": w(4096, 4096), "gate_up": w(28672, 4096), "down": w(4096, 14336)}])
    m.packed_lm = w(32000, 4096)
    assert all(m._slab_prompts(r) for r in (33, 48, 49, 96, 97, 128)) and all(m._wide(r) == (r > 96) for r in (33, 96, 97, 128))
    asked = []
    m._wide, m._slabs_pay = lambda r: asked.append(("wide", r)), lambda r: asked.append(("pay", r))
    for r in (96, 97):
        m._slab_prompts(r)
    assert asked == [("pay", 96), ("wide", 97)]


def test_rules_of_sizes_are_kept():
    """A step asks them of every layer's products."""
    for rule in (D.slab_split, D.wide_split, D.head_pays, D.slabs_fill):
        rule(100, 4096, 4096)
        hits = rule.cache_info().hits
        rule(100, 4096, 4096)
        assert rule.cache_info().hits == hits + 1
