"""Per-request state of many tensors moved in one launch (csrc/state_slots.hip)."""
from __future__ import annotations

from typing import List, Sequence

import ctypes

import torch

from . import _stream
from .library import KernelError, call, library


class StateSlots:
    """Tensors ``[slots, ...]`` that hold one row a request slot each, for clearing, copying and saving whole slots.  The table of
    their addresses lives as long as this object, which keeps the tensors alive."""

    ZERO, COPY, SAVE, RESTORE = range(4)

    def __init__(self, tensors: Sequence[torch.Tensor]):
        self.tensors = list(tensors)
        if not self.tensors:
            raise KernelError("state slots: no tensors")
        self.slots = self.tensors[0].shape[0]
        chunk, place, chunks, rows = library().leone_state_chunk(), 0, 0, []
        for t in self.tensors:
            if not self.takes(t) or t.shape[0] != self.slots or t.device != self.tensors[0].device:
                raise KernelError(f"state slots: cannot hold {tuple(t.shape)} {t.dtype} on {t.device} beside {self.slots} slots")
            size = t.stride(0) * t.element_size()
            rows.append((t.data_ptr(), size, place, chunks))
            place += (size + 15) // 16 * 16
            chunks += (size + chunk - 1) // chunk
        self.packed_bytes, self.chunks = place, chunks
        self.table = torch.tensor(rows, dtype=torch.int64, device=self.tensors[0].device)

    @staticmethod
    def takes(t) -> bool:
        """Whether a tensor can be among them: on the GPU, contiguous, rows of whole 4-byte words."""
        return (isinstance(t, torch.Tensor) and t.is_cuda and t.dim() >= 2 and t.is_contiguous() and t.numel() > 0
                and t.data_ptr() % 4 == 0 and t.stride(0) * t.element_size() % 4 == 0)

    def _move(self, move: int, ids: Sequence[int], to: Sequence[int] = (), packed=None) -> None:
        for slot in (*ids, *to):
            if not 0 <= slot < self.slots:
                raise KernelError(f"state slots: slot {slot} of {self.slots}")
        most = library().leone_state_slots_max()
        # On the tensors' device whatever the caller's is: requests are admitted and forked from any thread, and a thread that has
        # not chosen a device stands on the first.
        if torch.cuda.current_device() == self.table.device.index:
            self._launch(move, ids, to, packed, most)
        else:
            with torch.cuda.device(self.table.device):
                self._launch(move, ids, to, packed, most)

    def _launch(self, move: int, ids: Sequence[int], to: Sequence[int], packed, most: int) -> None:
        for at in range(0, len(ids), most):
            some, there = ids[at:at + most], to[at:at + most]
            array = ctypes.c_int * len(some)
            call("leone_state_slots", self.table.data_ptr(), len(self.tensors), self.chunks, move, array(*some),
                 array(*there) if there else None, len(some), 0 if packed is None else packed[at:].data_ptr(), self.packed_bytes, _stream())

    def zero(self, slots: Sequence[int]) -> None:
        self._move(self.ZERO, list(slots))

    def copy(self, from_slot: int, to_slot: int) -> None:
        if from_slot != to_slot:
            self._move(self.COPY, [from_slot], [to_slot])

    def save(self, slots: Sequence[int]) -> torch.Tensor:
        """What the slots hold, as packed rows for ``restore``."""
        packed = torch.empty((len(slots), self.packed_bytes), dtype=torch.uint8, device=self.table.device)
        if len(slots):
            self._move(self.SAVE, list(slots), packed=packed)
        return packed

    def restore(self, slots: Sequence[int], packed: torch.Tensor) -> None:
        if packed.shape != (len(slots), self.packed_bytes):
            raise KernelError(f"state slots: {tuple(packed.shape)} is not what {len(slots)} slots were saved as")
        if len(slots):
            self._move(self.RESTORE, list(slots), packed=packed)
