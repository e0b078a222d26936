"""Pinned host memory that launches read by its address."""
from __future__ import annotations

from typing import Optional

import torch


class PinnedBuffer:
    """`nbytes` of pinned memory for what launches of a step read.  torch knows of its own copies from pinned memory and keeps it until they have run; of a
    kernel's reads it does not, so this does: the memory is written again (wait()) or given back only once the last launch told of (read()) has run."""

    def __init__(self, nbytes: int):
        self.tensor = torch.empty(nbytes, dtype=torch.uint8, pin_memory=True)
        self._read: Optional[torch.cuda.Event] = None

    def wait(self) -> None:
        if self._read is not None:
            self._read.synchronize()

    def read(self) -> None:
        """Something on the current stream reads it."""
        self._read = torch.cuda.Event()
        self._read.record()

    def __del__(self):
        try:
            self.wait()
        except Exception:       # (the interpreter or the runtime is on its way out: so is the memory)
            pass
