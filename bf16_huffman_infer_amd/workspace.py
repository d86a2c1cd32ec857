"""Device workspaces of kernels whose blocks meet in memory: arrival counters, which a launch expects
to find at zero and leaves at zero, followed by partial results.

Launches that may overlap must not share one, so a workspace belongs to

* the (device, stream) of eager launches, which run one after the other, whichever threads enqueue them (the library
  enqueues the launches of one call in a row);
* the CAPTURE of recorded launches, not to the stream they were recorded on: graphs recorded one
  after the other on one stream (torch records every graph on the same one) may be replayed
  side by side, and none may depend on another having run first.

Under capture the memory comes from the graph's own pool and the counters are zeroed by a node of
the graph in front of the first launch that needs them, about 3 us of every replay.  A recorded
program that knows its needs beforehand has neither: :class:`Recording` notes what its warm-up runs
ask for and holds zeroed workspaces for the capture, for as long as the recorded program lives.
"""
import threading

import torch
from torch import Tensor

from . import _lib

_recording = threading.local()
_eager = {}             # (kind, device, stream) -> uint8 tensor
_captured = {}          # (kind, device, stream) -> (capture, uint8 tensor): the latest capture on that stream


class Recording:
    """The workspaces of one recorded program.  ``with recording.warmup():`` around the runs before the
    capture, ``with recording.capture():`` around the capture itself, on the same thread."""

    def __init__(self):
        self._needs = {}            # (kind, device) -> (bytes, counter bytes)
        self._held = {}             # (kind, device) -> tensor
        self._users = {}            # (kind, device) -> stream: a second stream of the capture gets its own

    class _Active:
        def __init__(self, recording):
            self.recording = recording

        def __enter__(self):
            self.outer = getattr(_recording, "current", None)
            _recording.current = self.recording

        def __exit__(self, *exc):
            _recording.current = self.outer

    def warmup(self):
        return Recording._Active(self)

    def capture(self):
        for (kind, device), (nbytes, counters) in self._needs.items():
            self._held[kind, device] = _fresh(device, nbytes, counters)
        torch.cuda.synchronize()    # zeroed before any stream replays the graph
        return Recording._Active(self)

    def _note(self, kind, device, nbytes, counters):
        old = self._needs.get((kind, device), (0, 0))
        self._needs[kind, device] = (max(nbytes, old[0]), max(counters, old[1]))

    def _take(self, kind, device, stream, nbytes):
        held = self._held.get((kind, device))
        if held is None or held.numel() < nbytes or self._users.setdefault((kind, device), stream) != stream:
            return None
        return held


def recorded() -> bool:
    """Whether the current call is being recorded into a graph, or is a warm-up run of a program that will be."""
    return getattr(_recording, "current", None) is not None or torch.cuda.is_current_stream_capturing()


def _fresh(device, nbytes, counters) -> Tensor:
    ws = torch.empty(nbytes, dtype=torch.uint8, device=device)
    ws[:counters].view(torch.int32).zero_()
    return ws


def capture_id(stream: int) -> int:
    """Nonzero and unique per capture while ``stream`` is being captured, else 0."""
    return int(_lib.load().bhi_stream_capture_id(stream))


def captured(kind: str, device: torch.device, stream: int, nbytes: int, counters: int):
    """The workspace for a launch under capture on ``stream``; None where nothing is being captured."""
    recording = getattr(_recording, "current", None)
    capture = capture_id(stream)
    if capture == 0:
        if recording is not None:
            recording._note(kind, device, nbytes, counters)
        return None
    if recording is not None:
        ws = recording._take(kind, device, stream, nbytes)
        if ws is not None:
            return ws
    key = (kind, device, stream)
    held = _captured.get(key)
    if held is None or held[0] != capture or held[1].numel() < nbytes:
        held = _captured[key] = (capture, _fresh(device, nbytes, counters))
    return held[1]


def workspace(kind: str, device: torch.device, stream: int, nbytes: int, counters: int) -> Tensor:
    """At least ``nbytes`` whose first ``counters`` bytes are zero between launches, for a launch on
    ``stream`` of ``device`` (the current stream).  A workspace that is replaced by a larger one was only
    used on ``stream``, in whose order the allocator hands its memory on."""
    ws = captured(kind, device, stream, nbytes, counters)
    if ws is None:
        key = (kind, device, stream)
        ws = _eager.get(key)
        if ws is None or ws.numel() < nbytes:
            ws = _eager[key] = _fresh(device, nbytes, counters)
    return ws
