"""``EventHandle`` and ``EventOverlap`` with the reference's public interface (deep_ep/utils/event.py:17-123:
constructor arguments, ``current_stream_wait``, ``wait``, ``register_hook_after_wait``, call / context-manager
protocol), over HIP events through ``torch.cuda``.

How it is put together here: a ``_Marker`` is one recorded HIP event plus where it was recorded; a ``_Lease`` keeps
objects alive and tells torch's caching allocator which streams use which tensors.  ``EventHandle`` is a marker with
a public face, ``EventOverlap`` a marker, a lease and an optional hook.  The native host path makes leases of its own
(``_host.Lease``) and marks a stream by the value of a counter (``_host.Marker``), with the same methods but no event.
"""

from __future__ import annotations

from typing import Any, Callable, Optional, Tuple

import torch


def gpu_api():
    """The framework's device API (streams, events).  One seam, so host-logic tests can run on CPU."""
    return torch.cuda


def _index_of(device) -> int:
    return getattr(device, "index", device)


class _Marker:
    """A HIP event recorded on ``stream`` (the current one if None) of the current GPU."""

    __slots__ = ("gpu", "stream", "event")

    def __init__(self, stream=None):
        api = gpu_api()
        self.gpu = api.current_device()
        self.stream = stream if stream is not None else api.current_stream(self.gpu)
        if _index_of(getattr(self.stream, "device", self.gpu)) != self.gpu:
            raise RuntimeError("Cannot record an event on another GPU")
        self.event = api.Event()
        self.event.record(self.stream)

    @classmethod
    def _of(cls, counted):
        """A HIP event that completes when the counter value of ``_host.Marker`` ``counted`` is reached, neither earlier nor
        later: recorded on a stream of its own that waits for the value and for nothing else."""
        api = gpu_api()
        marker = cls.__new__(cls)
        marker.gpu, marker.stream, marker.event = counted.gpu, counted.stream, api.Event()
        side = api.Stream(device=marker.gpu)
        counted.wait(side)
        marker.event.record(side)
        return marker

    def hold_current_stream(self):
        """Makes the current stream of the marker's GPU wait for the event; returns that stream."""
        api = gpu_api()
        if api.current_device() != self.gpu:
            raise RuntimeError("Cannot wait for an event from another GPU")
        consumer = api.current_stream(self.gpu)
        self.event.wait(consumer)
        return consumer


class _Lease:
    """Objects kept alive until released; the device tensors among them are declared to the allocator as in use
    on every stream that ``touch`` names, so that their memory is not handed out again while a stream still works
    on it."""

    __slots__ = ("objects", "tensors", "gpu")

    def __init__(self, objects, gpu: int):
        self.objects, self.gpu = objects, gpu
        flat = objects if isinstance(objects, (tuple, list)) else (objects,)
        self.tensors = [t for t in flat if isinstance(t, torch.Tensor) and t.device.type != "cpu" and t.device.index == gpu]

    def touch(self, stream) -> None:
        """None: the current stream (markers of the native host path do not make an object of it)."""
        if stream is None and self.tensors:
            stream = gpu_api().current_stream(self.gpu)
        for tensor in self.tensors:
            tensor.record_stream(stream)


class EventHandle:
    """An event recorded at construction, on ``stream`` or on the current stream."""

    def __init__(self, stream: Any = None) -> None:
        self._marker = _Marker(stream)

    @property
    def event(self) -> Any:
        """The event itself, one of torch's.  From then on the handle goes by it (so recording it again counts)."""
        if not isinstance(self._marker, _Marker):
            self._marker = _Marker._of(self._marker)
        return self._marker.event

    @property
    def _gpu_index(self) -> int:
        """Index of the GPU the event was recorded on."""
        return self._marker.gpu

    def current_stream_wait(self) -> None:
        self._marker.hold_current_stream()


class EventOverlap:
    """An ``EventHandle`` together with what has to outlive the work it marks.

    ``EventOverlap()`` with no event is valid and has nothing to wait for.  ``with overlap: ...`` waits when the block
    ends; ``with overlap(release_handle=True): ...`` also drops the event and the retained objects then.
    """

    # (what an overlap without an event has; the native host path makes those without running __init__)
    event: Optional[EventHandle] = None
    extra_tensors: Optional[Tuple[torch.Tensor]] = None
    hook_after_wait: Optional[Callable] = None
    _lease: Optional[_Lease] = None
    _release_on_exit = False

    def __init__(self, event: Optional[EventHandle] = None, extra_tensors: Optional[Tuple[torch.Tensor]] = None) -> None:
        self.event = event
        self.extra_tensors = extra_tensors
        self.hook_after_wait: Optional[Callable] = None
        self._lease: Optional[_Lease] = None
        self._release_on_exit = False
        if isinstance(event, EventHandle) and extra_tensors is not None:
            self._take(extra_tensors)

    def _take(self, objects) -> None:
        marker = self.event._marker
        self._lease = _Lease(objects, marker.gpu)
        self._lease.touch(marker.stream)  # the producer stream is still working on them

    @classmethod
    def _holding(cls, event: EventHandle, objects: Tuple[Any, ...]) -> "EventOverlap":
        """An overlap that keeps ``objects`` (tensors and anything else) alive until it is waited on with
        ``release_handle=True`` or dropped."""
        overlap = cls(event)
        overlap._take(objects)
        return overlap

    def current_stream_wait(self, release_handle: bool = False) -> Any:
        assert self.event is not None
        consumer = self.event._marker.hold_current_stream()
        if self._lease is not None:
            self._lease.touch(consumer)
        hook, self.hook_after_wait = self.hook_after_wait, None
        outcome = hook() if hook is not None else None
        if release_handle:
            self.event = None
            self._lease = None
        return outcome

    def wait(self) -> Any:
        return self.current_stream_wait()

    def register_hook_after_wait(self, hook_after_wait: Callable) -> None:
        assert self.hook_after_wait is None, "A hook is already registered on this `EventOverlap`"
        self.hook_after_wait = hook_after_wait

    def __call__(self, release_handle: bool = False) -> "EventOverlap":
        self._release_on_exit = release_handle
        return self

    def __enter__(self) -> Any:
        return self

    def __exit__(self, exc_type: Any, exc_val: Any, exc_tb: Any) -> None:
        release, self._release_on_exit = self._release_on_exit, False
        if self.event is not None:
            self.current_stream_wait(release_handle=release)
