"""Caller-side workspaces for the multi-launch kernels.

The C-ABI allocates nothing.  Intermediate records (the expert's act vector, router
records, split-T partials, grouping lists) live in a workspace the caller passes in.
Concurrent launches must not share a workspace, so workspaces are kept per (device,
stream, user, thread): the launches of two threads' calls may interleave on one stream.  (A
later thread may get an ended one's number, and with it its buffers; on one stream that is
in order.  The prompt paths allocate their scratch per call instead.)

A captured graph goes on using the buffer its capture was given.  So a buffer that a later call
outgrows is kept beside its successor, which is at least twice as large, so all of one key's outgrown
buffers are smaller than the one in use; and a call inside a capture that finds no buffer gets one
of that capture's own, its counters cleared by a node of the graph: buffers made in a capture are
not shared with other captures or eager calls, which may run before that graph ever does.
``clear`` gives everything back; it is for programs that hold no captured graph.
"""
from __future__ import annotations

import threading

import torch

from . import _lib
from . import _torch as T

COUNTERS = 4096      # bytes at the head of a workspace that some kernels want zeroed once

_lock = threading.Lock()
_cache: dict[tuple, torch.Tensor] = {}
_outgrown: list[torch.Tensor] = []
_captured: dict[tuple, tuple[int, torch.Tensor]] = {}    # (capture, its buffer)


def get(device: torch.device, nbytes: int, tag: str = "") -> torch.Tensor:
    """A uint8 device buffer of at least nbytes for the current stream and thread, zero when made
    (inside a capture: its first COUNTERS bytes)."""
    key = (device.index, T.stream_of(device), tag, threading.get_ident())
    buf = _cache.get(key)
    if buf is None or buf.numel() < nbytes:
        buf = _make(device, nbytes, key)
    return buf


def _make(device: torch.device, nbytes: int, key: tuple) -> torch.Tensor:
    nbytes = max(nbytes, COUNTERS)
    capture = _lib.lib().k3_stream_capture_id(key[1])
    with _lock:
        if capture:
            made, buf = _captured.get(key, (0, None))
            if made != capture or buf.numel() < nbytes:
                buf = torch.empty(nbytes, dtype=torch.uint8, device=device)
                buf[:COUNTERS].zero_()
                _captured[key] = (capture, buf)
            return buf
        old = _cache.get(key)
        if old is not None and old.numel() >= nbytes:
            return old
        if old is not None:
            _outgrown.append(old)
            nbytes = max(nbytes, 2 * old.numel())
        buf = _cache[key] = torch.zeros(nbytes, dtype=torch.uint8, device=device)
    return buf


def clear() -> None:
    with _lock:
        _cache.clear()
        _captured.clear()
        _outgrown.clear()
