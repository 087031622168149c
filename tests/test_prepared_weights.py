"""The packed weights that the layer functions keep between calls: CPU checks
of when a call packs (preparation and launches replaced by stand-ins)."""

import pytest
import torch

from smolvla import layers
from smolvla.config import VitConfig
from smolvla.vla import _common, vision_block_bf16


@pytest.fixture
def packs(monkeypatch):
    """vision_block on CPU tensors, its launches left out; returns the calls
    of prep_vit."""
    calls = []

    def prep(p, device, rows=None):
        calls.append(rows)
        return dict(p)

    monkeypatch.setattr(vision_block_bf16, "to_device", lambda x: (x, lambda t: t))
    monkeypatch.setattr(layers, "prep_vit", prep)
    monkeypatch.setattr(layers, "vit_layer", lambda *a, **k: None)
    return calls


def test_vision_block_packs_once_for_every_size(packs):
    """No call size may find its weights unpacked after a call of another: it
    may come inside a graph capture, where packing would only be recorded."""
    params = {"Wq": torch.zeros(8, 768), "W_up": torch.zeros(8, 3072)}
    for rows in (196, 4 * 1024, 1024, 12 * 1024, 96 * 1024 + 64):
        x = torch.empty(1, rows, 768, dtype=torch.bfloat16)
        vision_block_bf16.vision_block(x, params, VitConfig())
    assert len(packs) == 1


@pytest.mark.parametrize("hidden,inter", [(768, 3072), (768, 384), (1152, 4304), (128, 256)])
def test_blockable_is_the_plan_at_large_calls(hidden, inter):
    fits = layers.vit_blockable(hidden, inter)
    assert fits == layers.vit_blocked_plan(hidden, inter, 256 * layers.WIDE_MIN_TILES)
    for rows in (256, 3072, 4096, 12288, 12300):
        plan = layers.vit_blocked_plan(hidden, inter, rows)
        assert all(fits[k] or not plan[k] for k in plan)


def test_what_a_capture_packs_is_not_kept(monkeypatch):
    """Packing inside a graph capture is recorded, not run: a later call may
    not take its tensors for packed weights, nor lose an entry to them."""
    calls = []
    pack = lambda p, device: calls.append(p) or len(calls)  # noqa: E731
    params, kept = {"W": torch.ones(2)}, {"W": torch.zeros(2)}
    assert _common.prepared(kept, pack) == 1
    monkeypatch.setattr(_common, "_capturing", lambda: True, raising=False)
    assert _common.prepared(params, pack) == 2
    assert _common.prepared(params, pack) == 3              # one graph's, not another's
    assert _common.prepared(kept, pack) == 1                # packed before: used as it is
    monkeypatch.setattr(_common, "_capturing", lambda: False, raising=False)
    assert _common.prepared(params, pack) == 4              # an eager call packs its own
    assert _common.prepared(params, pack) == 4 and len(calls) == 4


class _Stream:
    def __init__(self):
        self.waited = []

    def wait_event(self, event):
        self.waited.append(event)


class _Event:
    def record(self):
        self.stream = torch.cuda.current_stream()


def test_another_stream_waits_for_the_packing(monkeypatch):
    """The first hit on another stream than the one that packed waits for the
    packing; a hit inside a capture does not."""
    here, there, third = _Stream(), _Stream(), _Stream()
    cur = [here]
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: cur[0])
    monkeypatch.setattr(_common, "_raw_stream", lambda: id(cur[0]), raising=False)
    monkeypatch.setattr(torch.cuda, "Event", _Event)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    recorded = []
    monkeypatch.setattr(torch.Tensor, "record_stream", lambda t, s: recorded.append((t, s)))
    params, w = {"W": torch.ones(2)}, torch.ones(3)
    pack = lambda p, device: dict(w=w, b=None)  # noqa: E731
    _common.prepared(params, pack)
    _common.prepared(params, pack)
    assert not here.waited and not recorded
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    cur[0] = there
    _common.prepared(params, pack)
    assert not there.waited
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    for _ in range(2):
        _common.prepared(params, pack)
    assert [e.stream for e in there.waited] == [here]
    assert len(recorded) == 1 and recorded[0][0] is w and recorded[0][1] is there
    cur[0] = third
    _common.prepared(params, pack)
    assert [e.stream for e in third.waited] == [here] and len(recorded) == 2
    assert not here.waited
