"""The gradient table apply_gradient builds from a per-name dict: what goes to
the fused path, what falls back to the per-name copies, and that every layout a
gradient can have ends up in the same columns (CPU key)."""

from __future__ import annotations

from collections import OrderedDict
from types import MappingProxyType

import pytest
import torch
from torch.autograd import forward_ad

import churten_amd.kernels  # noqa: F401
from churten_amd.optimizer import SGD
from churten_amd.state import State

SHAPES = {"a": (3, 2), "b": (3,), "c": (2, 3, 2), "d": ()}


def make(meta_type=torch.Size, dtype=torch.float32):
    meta, off = [], 0
    for name, s in SHAPES.items():
        n = int(torch.Size(s).numel())
        meta.append((name, meta_type((4, *s)), off, n))
        off += n
    T = off + (-off % 4)
    p = torch.arange(4 * T, dtype=dtype).reshape(4, T)
    state = State(params=p, buffers=torch.empty(4, 0), param_meta=meta, buffer_meta=[])
    return SGD.init(state, lr=0.5)


def grads_of(dtype=torch.float32):
    g = torch.Generator().manual_seed(4)
    return {k: torch.randn(4, *s, generator=g).to(dtype) for k, s in SHAPES.items()}


def consolidated(grads, T):
    out = torch.zeros(4, T)
    off = 0
    for k, s in SHAPES.items():
        n = int(torch.Size(s).numel())
        out[:, off:off + n] = grads[k].detach().reshape(4, n)
        off += n
    return out


def strided(t):
    wide = torch.zeros(*t.shape[:-1], 2 * t.shape[-1])
    wide[..., ::2] = t
    return wide[..., ::2]


LAYOUTS = {
    "contiguous": lambda k, t: t,
    "requires_grad": lambda k, t: t.clone().requires_grad_(),
    "row_strided": lambda k, t: torch.cat([t[:, None], t[:, None]], dim=1)[:, 0],
    "inner_strided": lambda k, t: strided(t) if t.dim() > 1 else t,
    "transposed": lambda k, t: t.transpose(0, -1).contiguous().transpose(0, -1),
    "expanded": lambda k, t: t[:1].expand(t.shape),
}


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("order", [1, -1])
@pytest.mark.parametrize("meta_type", [torch.Size, list, tuple])
def test_layouts(layout, order, meta_type):
    state = make(meta_type)
    grads = {k: LAYOUTS[layout](k, t) for k, t in list(grads_of().items())[::order]}
    before = state.params.clone()
    want = consolidated(grads, state.params.shape[1])
    SGD.apply_gradient(state, grads)
    assert torch.equal(state.grads, want)
    assert torch.equal(state.params, before - 0.5 * want)


def test_what_falls_back():
    state = make()
    table = state._consolidated_grads.segments
    full = grads_of()
    assert table(full)[1] == [0, 6, 9, 21]
    assert table({"c": full["c"]})[1] == [9]  # part of the names
    assert table({}) == ([], [])
    for bad in ({"zz": full["a"]}, {"a": full["a"], "zz": full["b"]}, {"a": None},
                {"a": full["a"].double()}, {"a": full["a"][:3]}, {"a": full["a"][0]},
                {"a": full["a"].reshape(4, 6)}, {"a": 1.0}):
        assert table(bad) is None


def test_unknown_name_is_refused_and_views_still_alias():
    state = make()
    grads = grads_of()
    with pytest.raises(KeyError):
        SGD.apply_gradient(state, {**{k: grads[k] for k in "abc"}, "zz": grads["d"]})
    view = state._consolidated_grads
    assert list(view.keys()) == list(SHAPES)
    view["b"].fill_(2.0)
    assert bool((state.grads[:, 6:9] == 2.0).all())


class ItemsOnly:
    """A mapping of which only items() and the length are there."""

    def __init__(self, d):
        self._d = d

    def __len__(self):
        return len(self._d)

    def items(self):
        return self._d.items()


@pytest.mark.parametrize("kind", [ItemsOnly, MappingProxyType, OrderedDict])
@pytest.mark.parametrize("names", ["abcd", "ac"])
def test_mappings(kind, names):
    state, other = make(), make()
    grads = {k: g for k, g in grads_of().items() if k in names}
    SGD.apply_gradient(state, kind(grads))
    SGD.apply_gradient(other, grads)
    assert torch.equal(state.params, other.params)
    assert torch.equal(state.grads, other.grads) and bool(state.grads.any())


@pytest.mark.parametrize("names", ["abcd", "ac"])
def test_dual_gradients_leave_no_tangent(names):
    """The state is plain data: a forward-mode gradient's tangent does not get
    into its buffers."""
    state, other = make(), make()
    grads = {k: g for k, g in grads_of().items() if k in names}
    with forward_ad.dual_level():
        SGD.apply_gradient(state, {k: forward_ad.make_dual(g, torch.ones_like(g))
                                   for k, g in grads.items()})
        for t in (state.params, state.grads):
            assert forward_ad.unpack_dual(t).tangent is None
    SGD.apply_gradient(other, grads)
    assert torch.equal(state.params, other.params) and torch.equal(state.grads, other.grads)


@pytest.mark.parametrize("bad", [("a", (4, 3, 2), 0, 5), ("b", (4, 3), 6, 4)])
@pytest.mark.parametrize("given", ["all", "others"])
def test_metadata_that_contradicts_itself_is_refused(bad, given):
    """A width that is not the shape's would write the gradient's own width over
    the next parameter's columns."""
    state = make()
    state.param_meta = [bad if m[0] == bad[0] else m for m in state.param_meta]
    grads = grads_of()
    if given == "others":
        del grads[bad[0]]
    before = state.params.clone()
    with pytest.raises(RuntimeError):
        SGD.apply_gradient(state, grads)
    assert torch.equal(state.params, before) and not state.grads.any()


@pytest.mark.parametrize("meta_type", [torch.Size, list])
def test_metadata_changed_after_a_step_is_noticed(meta_type):
    """What was found to agree once is compared by content, not by identity."""
    state = make(meta_type)
    grads = grads_of()
    SGD.apply_gradient(state, grads)
    good = state.param_meta[0]
    if meta_type is list:
        good[1][2] = 1  # the list inside the entry
    else:
        state.param_meta[0] = (good[0], good[1], good[2], 5)
    with pytest.raises(RuntimeError):
        SGD.apply_gradient(state, grads)
    if meta_type is list:
        good[1][2] = 2
    else:
        state.param_meta[0] = good
    SGD.apply_gradient(state, grads)
    state.grads = state.grads[:3].clone()  # rows that the metadata does not have
    with pytest.raises(RuntimeError):
        SGD.apply_gradient(state, grads)
