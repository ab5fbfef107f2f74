"""The streams of batches that run at once.

A library keeps the workspace of its products by the stream that they are launched or recorded on, and a captured graph keeps
the workspace it was recorded with.  So two batches may be under way at once only if no stream that one of them is recorded,
warmed up or forked on is one of the other's.  Torch's streams come from a pool of a few dozen that hands them out in turn:
whoever draws a new one for a moment gets, sooner or later, one that a graph was recorded on.  The streams of every kind of
batch are therefore drawn once a device, each of them another one than all the others, and a fork's second stream is
found by the stream that it forks from."""
from __future__ import annotations

import threading
from typing import Callable, Dict, Optional

import torch

# kinds of captured steps: the graphs of two kinds may run at once, those of one kind follow each other
SINGLES, PORTIONS, SECOND_HALF = "single tokens", "portions", "second half of the single tokens"
KINDS = (SINGLES, PORTIONS, SECOND_HALF)

# The runtime lays its streams on a few hardware queues (four by default), in turn, and what lies on one queue runs one after
# the other: streams drawn in a row, one more than may stand in the way of the caller's.
BESIDE_STREAMS = 5


class BatchStreams:
    """``recording[kind]``: the stream that graphs of the kind are recorded on; ``side[kind]``: the stream that they fork their
    first mixer to; ``beside``: streams that a graph may be replayed on beside the caller's stream.  What runs ahead of a
    recording, or forks elsewhere, is on a stream ``apart`` from all of these."""

    def __init__(self, draw: Callable, usual: Optional["torch.cuda.Stream"] = None):
        """``draw()``: a stream, perhaps one that is taken.  ``usual``: the stream that torch records graphs on by default."""
        self._draw = draw
        self._taken = []
        self.recording, self.side = {}, {}
        self.forks = dict.fromkeys(KINDS, 0)             # how often a recording of the kind took its second stream
        if usual is not None:
            self.recording[SINGLES] = usual
            self._taken.append(usual)
        for kind in KINDS:
            for streams in (self.recording, self.side):
                if kind not in streams:
                    streams[kind] = self.apart()
                    self._taken.append(streams[kind])
        self.beside = []
        for _ in range(BESIDE_STREAMS):
            self.beside.append(self.apart())
            self._taken.append(self.beside[-1])

    def apart(self) -> "torch.cuda.Stream":
        """A stream that is none of these."""
        while True:
            stream = self._draw()
            if all(stream != other for other in self._taken):
                return stream

    def side_of(self, main: "torch.cuda.Stream") -> Optional["torch.cuda.Stream"]:
        """The stream that work recorded on ``main`` forks to (None: no kind of batch is recorded there)."""
        for kind in KINDS:
            if main == self.recording[kind]:
                return self.side[kind]
        return None

    def fork(self, main: "torch.cuda.Stream") -> Optional["torch.cuda.Stream"]:
        """``side_of(main)`` for work that is recorded there now."""
        for kind in KINDS:
            if main == self.recording[kind]:
                self.forks[kind] += 1
        return self.side_of(main)

    def belongs_to(self, kind: str, stream: "torch.cuda.Stream") -> bool:
        return stream == self.recording[kind] or stream == self.side[kind]


_of_device: Dict[int, BatchStreams] = {}
_lock = threading.Lock()


def batch_streams(device: torch.device) -> BatchStreams:
    """The streams of the device (default priority)."""
    index = device.index if device.index is not None else torch.cuda.current_device()
    with _lock:
        if index not in _of_device:
            draw = lambda: torch.cuda.Stream(device=torch.device("cuda", index))
            usual = torch.cuda.graph.default_capture_stream
            if usual is None:
                usual = torch.cuda.graph.default_capture_stream = draw()
            _of_device[index] = BatchStreams(draw, usual if usual.device.index == index else None)
        return _of_device[index]
