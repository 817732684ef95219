"""Workspaces of prepared calls that may be launched on several streams."""

from __future__ import annotations

import torch

_is_capturing = torch._C._cuda_isCurrentStreamCapturing


class StreamWorkspaces:
    """The workspaces of one prepared call: one per stream that launches it,
    so launches in flight on several streams (or threads, each on its own)
    do not meet in one.  A launch under capture gets one of its own, since
    its graph may be replayed on any stream.  Those of graphs are kept, as the
    graph needs them, as long as the call; of the streams', the last
    ``STREAMS`` new ones (an older stream's next launch allocates again: it
    is freed to its own stream's later allocations, behind what runs there)."""

    STREAMS = 32

    def __init__(self, before: tuple, first: torch.Tensor, after: tuple, stream: int):
        """before, after: the library call's arguments around the workspace's
        address; the stream follows them.  first: ``stream``'s workspace."""
        self._before, self._after = before, after
        self._device, self._bytes = first.device, first.numel()
        self._by_stream = {stream: self._entry(first, stream)}
        self._captured = []
        self._elsewhere = torch.cuda.device_count() > 1  # another device may be the current one

    def _entry(self, ws: torch.Tensor, stream: int) -> tuple:
        return (*self._before, ws.data_ptr(), *self._after, stream), ws

    def _new(self, stream: int) -> tuple:
        return self._entry(torch.empty(self._bytes, dtype=torch.uint8, device=self._device), stream)

    def _capturing(self) -> bool:
        if self._elsewhere and torch.cuda.current_device() != self._device.index:
            with torch.cuda.device(self._device):
                return _is_capturing()
        return _is_capturing()

    def on(self, stream: int) -> tuple:
        """(library arguments, workspace) of a launch on ``stream``, the
        device's current one; the caller holds the workspace until it has
        launched."""
        if self._capturing():
            entry = self._new(stream)
            self._captured.append(entry)
            return entry
        entry = self._by_stream.get(stream)
        if entry is None:
            entry = self._by_stream.setdefault(stream, self._new(stream))
            if len(self._by_stream) > self.STREAMS:
                self._by_stream.pop(next(iter(self._by_stream)), None)
        return entry
