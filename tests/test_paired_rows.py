"""Who is handed routed experts' results that are still to be summed over their places."""
import gc
import weakref
from types import SimpleNamespace

import pytest
import torch

from leone_amd import ops
from leone_amd.parts.block import PostNormBlock
from leone_amd.parts.feedforward import RoutedGluMlp
from leone_amd.parts.norm import RmsNorm

STEP = SimpleNamespace(dtype=torch.float32)


def _block(norm, feed_forward):
    block = PostNormBlock.__new__(PostNormBlock)
    block.mixer = SimpleNamespace(forward=lambda h, step, cache: h)
    block.norm1 = SimpleNamespace(add_behind=lambda x, delta, kind: x)
    block.norm2, block.feed_forward = norm, feed_forward
    return block


def _pairs(monkeypatch):
    pairs = ops.PairedRows(torch.ones(4, 3), None, None, torch.zeros(2, 3), None, 1)
    monkeypatch.setattr(ops.PairedRows, "sum", lambda self: self.pairs.view(2, 2, 3).sum(1))
    monkeypatch.setattr(ops, "routed_feed_forward", lambda *args, paired=False, **kwargs: pairs if paired else pairs.sum())
    monkeypatch.setattr(ops, "linear", lambda y, *args, **kwargs: y)
    return pairs


def _routed(kind=RoutedGluMlp):
    part = kind.__new__(kind)
    part.__dict__.update(w_router=None, always=0, shared=None, correction=None, top=2, group_count=1, group_keep=1, w_gate_up=None, w_down=None,
                         activation="silu", rule=None, limit=None, weigh_input=False)
    return part


@pytest.mark.parametrize("own", ["class", "subclass", "object"])
def test_a_norm_of_its_own_gets_the_sum(monkeypatch, own):
    """A norm that stands behind a sublayer in another way, whatever way it took the place of the ordinary one's method."""
    seen = []

    def add_behind(x, delta, kind):
        seen.append(delta)
        return x

    class Own:
        def add_behind(self, x, delta, kind):
            return add_behind(x, delta, kind)

    class Sub(RmsNorm):
        def add_behind(self, x, delta, kind):
            return add_behind(x, delta, kind)

    norm = Own() if own == "class" else Sub.__new__(Sub) if own == "subclass" else RmsNorm.__new__(RmsNorm)
    if own == "object":
        norm.add_behind = add_behind
    _pairs(monkeypatch)
    pending = ops.NormedDelta(_routed().forward(torch.zeros(2, 3), STEP, paired=True), norm)
    PostNormBlock._take_in(torch.zeros(2, 3), pending, STEP)
    assert len(seen) == 1 and torch.equal(seen[0], torch.full((2, 3), 2.0))
    assert torch.equal(pending.rows, seen[0])


def test_the_ordinary_norm_gets_the_places(monkeypatch):
    pairs, seen = _pairs(monkeypatch), []
    monkeypatch.setattr(ops, "add_normed", lambda x, delta, *args, **kwargs: seen.append(delta) or x)
    norm = RmsNorm.__new__(RmsNorm)
    norm.groups, norm.gain, norm.eps = 1, torch.ones(3), 1e-5
    block = _block(norm, _routed())
    pending = block.forward(torch.zeros(2, 3), None, STEP, None)
    seen.clear()
    block._take_in(torch.zeros(2, 3), pending, STEP)
    assert seen == [pairs]


@pytest.mark.parametrize("where", ["block", "norm"])
def test_places_are_let_go_once_they_are_in_the_stream(monkeypatch, where):
    """Whoever still holds the delta, as the model and the block do until the block returns, holds no places with it."""
    norm = RmsNorm.__new__(RmsNorm)
    norm.groups, norm.gain, norm.eps = 1, torch.ones(3), 1e-5
    pending = ops.NormedDelta(ops.PairedRows(torch.ones(4, 3), None, None, torch.zeros(2, 3), None, 1), norm)
    monkeypatch.setattr(ops, "add_normed", lambda x, delta, *args, **kwargs: x)
    places = weakref.ref(pending.unsummed.pairs)
    if where == "block":
        PostNormBlock._take_in(torch.zeros(2, 3), pending, STEP)
    else:
        assert norm.add_norm(torch.zeros(2, 3), pending, torch.float32, torch.tensor([0])) is not None and places() is not None   # nothing added yet
        norm.add_norm(torch.zeros(2, 3), pending, torch.float32)
    gc.collect()
    assert places() is None
    with pytest.raises(ops.KernelError):
        pending.rows


def test_a_feed_forward_of_its_own_is_called_as_ever(monkeypatch):
    class Sub(RoutedGluMlp):
        def forward(self, y, step):
            return super().forward(y, step) * 3

    _pairs(monkeypatch)
    monkeypatch.setattr(ops, "add_normed", lambda x, delta, *args, **kwargs: x)
    pending = _block(SimpleNamespace(add_behind=None), _routed(Sub)).forward(torch.zeros(2, 3), None, STEP, None)
    assert torch.equal(pending.rows, torch.full((2, 3), 6.0))
