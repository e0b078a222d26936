"""Pinned host memory that launches read by its address."""
from __future__ import annotations

from typing import List, Optional, Tuple

import torch

_kept: List[Tuple[torch.cuda.Event, torch.Tensor]] = []      # what could not be waited for when its buffer went, until it has been read


class PinnedBuffer:
    """`nbytes` of pinned memory for what launches of a step read.  torch knows of its own copies from pinned memory and keeps it until they have run; of a
    kernel's reads it does not, so this does: the memory is written again (wait()) or given back only once the last launch told of (read()) has run."""

    def __init__(self, nbytes: int):
        self._read: Optional[torch.cuda.Event] = None
        if _kept and not torch.cuda.is_current_stream_capturing():
            _kept[:] = [k for k in _kept if not k[0].query()]
        self.tensor = torch.empty(nbytes, dtype=torch.uint8, pin_memory=True)

    def wait(self) -> None:
        if self._read is not None:
            self._read.synchronize()

    def read(self) -> None:
        """Something on the current stream reads it."""
        self._read = torch.cuda.Event()
        self._read.record()

    def __del__(self):
        if self._read is None:
            return
        try:
            if not torch.cuda.is_current_stream_capturing():      # (a wait would end the capture)
                return self.wait()
        except Exception:       # (the runtime is on its way out, or does not let us wait here)
            pass
        if _kept is not None:      # (a module being torn down)
            _kept.append((self._read, self.tensor))
