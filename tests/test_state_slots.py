"""Where the launch that moves request slots goes."""
from contextlib import contextmanager
from types import SimpleNamespace

import pytest
import torch


@pytest.mark.parametrize("move", ["zero", "copy", "save", "restore"])
def test_slots_move_on_their_tensors_device(monkeypatch, move):
    """Requests are admitted and forked from threads that stand on another device than the engine's."""
    from leone_amd.ops import state
    current, seen = ["cuda:0"], []

    @contextmanager
    def device(of):
        before, current[0] = current[0], str(of)
        yield
        current[0] = before

    monkeypatch.setattr(torch.cuda, "device", device)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: int(current[0][-1]))
    monkeypatch.setattr(state, "library", lambda: SimpleNamespace(leone_state_slots_max=lambda: 64))
    monkeypatch.setattr(state, "_stream", lambda: current[0])
    monkeypatch.setattr(state, "call", lambda name, *args: seen.append(args[-1]))
    held = state.StateSlots.__new__(state.StateSlots)
    held.tensors, held.slots, held.chunks, held.packed_bytes = [None], 8, 1, 16
    held.table = SimpleNamespace(device=torch.device("cuda:1"), data_ptr=lambda: 0)
    packed = torch.zeros(2, 16, dtype=torch.uint8)
    monkeypatch.setattr(torch, "empty", lambda *args, **kwargs: packed)
    {"zero": lambda: held.zero([1]), "copy": lambda: held.copy(1, 2), "save": lambda: held.save([1, 2]),
     "restore": lambda: held.restore([1, 2], packed)}[move]()
    assert seen == ["cuda:1"] and current == ["cuda:0"]
