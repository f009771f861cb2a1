"""Values derived from a few tensors (a stack of weights, scaled random matrices), kept until one
of the tensors changes.

An entry remembers, for every source tensor, a weak reference to the tensor object and its version
counter, storage address, dtype, shape, strides and device.  It answers only for the very same objects in the
very same state: an in-place update moves the version counter, ``p.data = ...`` moves the address (or, for a
view of the same storage, the strides), and a tensor that has died cannot be impersonated by a new one
that the allocator put at its address (or that Python gave its id), because the weak reference is dead.

A value is also tied to the stream that made it: a caller on another stream has nothing that would make
its kernels wait for that one, and memory that an entry gives back may be used again by its own
stream at once.  While a stream is captured nothing is kept and nothing kept is used: what the graph reads must
live as long as the graph, and be formed from the tensors of the day at each replay.
"""
from __future__ import annotations

import weakref
from typing import Callable, Optional, Sequence

import torch
from torch import Tensor

from . import rfa_hip


def _stream(sources: Sequence[Optional[Tensor]]) -> Optional[int]:
    """Handle of the stream that work on these tensors is issued to (0: the default one, which cannot be captured, or no
    device tensor), None while it is captured."""
    for t in sources:
        if t is not None and t.is_cuda:
            stream = rfa_hip._stream_ptr(t.device)
            return None if stream and torch.cuda.is_current_stream_capturing() else stream
    return 0


def _state(t: Optional[Tensor]):
    return None if t is None else (t._version, t.data_ptr(), t.dtype, t.shape, t.stride(), t.device)


class _Entry:
    __slots__ = ("refs", "state", "extra", "value")

    def __init__(self, sources, state, extra, value):
        self.refs = tuple(None if t is None else weakref.ref(t) for t in sources)
        self.state, self.extra, self.value = state, extra, value

    def answers(self, sources, state, extra) -> bool:
        if self.state != state or self.extra != extra or len(self.refs) != len(sources):
            return False
        return all((r is None and t is None) or (r is not None and t is not None and r() is t)
                   for r, t in zip(self.refs, sources))

    def alive(self) -> bool:
        return all(r is None or r() is not None for r in self.refs)


def derived(slot: dict, name, sources: Sequence[Optional[Tensor]], extra, make: Callable, limit: int = 0):
    """``make()`` for these source tensors, from ``slot[name]`` if that entry was made from the same
    tensor objects in the same state (and the same ``extra``), else made and stored there; on another stream
    than the default one under (name, stream).  With ``limit`` > 0 the slot is first cleared of entries whose
    sources have died and, if it is still that full, emptied."""
    stream = _stream(sources)
    if stream is None:
        return make()
    if stream:
        name = (name, stream)
    state = tuple(_state(t) for t in sources)
    e = slot.get(name)
    if e is not None and e.answers(sources, state, extra):
        return e.value
    value = make()
    if limit and len(slot) >= limit and name not in slot:
        for k in [k for k, v in slot.items() if not v.alive()]:
            del slot[k]
        if len(slot) >= limit:
            slot.clear()
    slot[name] = _Entry(sources, state, extra, value)
    return value
