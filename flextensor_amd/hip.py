"""Streams, events and host arenas over the C ABI.

:class:`HipStream` wraps a ``hipStream_t`` (normally the handle of a
``torch.cuda.Stream``) and offers the ``record_event / wait_event /
wait_stream / synchronize`` surface the transfer runtime uses, in the
shape the reference uses PyTorch's stream objects (core/transfer.py:49-146).
:class:`HostArena` is one page-locked, device-mapped host allocation exposed
as a CPU ``uint8`` tensor without copying.
"""

from __future__ import annotations

import ctypes
from collections.abc import Iterator
from contextlib import contextmanager
from typing import Any

import torch

from . import _native as nat


_FREE_EVENTS: dict[int, list[int]] = {}  # recycled handles by creation flags
_MAX_FREE_EVENTS = 4096


class HipEvent:
    """One ``hipEvent_t``.

    Handles are recycled through a free list instead of being destroyed: the
    streaming loop creates and drops several events per label, and an event
    dropped by Python may still be pending on a stream. Re-recording a
    recycled handle is safe because a wait always refers to the record that
    preceded it.
    """

    __slots__ = ("handle", "timing", "flags", "__weakref__")

    def __init__(self, timing: bool = False, device_only: bool = False) -> None:
        """``device_only``: only streams of this device wait on it, so recording it skips the system-scope
        fence (``FTX_EVENT_DEVICE_ONLY``); host waits still see it complete."""
        self.timing = timing
        self.flags = (nat.EVENT_TIMING if timing else nat.EVENT_DEFAULT) | (nat.EVENT_DEVICE_ONLY if device_only else 0)
        free = _FREE_EVENTS.setdefault(self.flags, [])
        self.handle = free.pop() if free else nat.event_create(self.flags)

    def record(self, stream: "HipStream | None" = None) -> "HipEvent":
        s = stream if stream is not None else current_stream()
        nat.call("ftx_event_record", self.handle, s.handle)
        return self

    def query(self) -> bool:
        return nat.event_query(self.handle)

    def synchronize(self) -> None:
        nat.call("ftx_event_synchronize", self.handle)

    def elapsed_time(self, end: "HipEvent") -> float:
        return nat.event_elapsed_ms(self.handle, end.handle)

    def __del__(self) -> None:
        h = getattr(self, "handle", None)
        if not h:
            return
        self.handle = None
        try:
            if not nat.live():
                return
            free = _FREE_EVENTS.setdefault(self.flags, [])
            if len(free) < _MAX_FREE_EVENTS:
                free.append(h)
            else:
                nat.lib().ftx_event_destroy(h)
        except (TypeError, AttributeError):
            pass  # interpreter shutdown: module globals are already gone; the process frees the handle


class DeviceClock:
    """A device array of wall-clock timestamps written by ``ftx_timestamp``.

    Its events are kernel launches, so a graph that captures them writes new
    times on every replay. :meth:`refresh` copies the array to the host once
    the device is idle; elapsed times are then read from that copy.
    """

    def __init__(self, n: int, device: torch.device | int | None = None) -> None:
        dev = torch.device("cuda", torch.cuda.current_device()) if device is None else torch.device(device)
        self.buf = torch.zeros(max(1, n), dtype=torch.int64, device=dev)
        self.host: list[int] = [0] * max(1, n)
        khz = ctypes.c_int(0)
        nat.call("ftx_wall_clock_khz", ctypes.byref(khz))
        if khz.value <= 0:
            raise RuntimeError("the device reports no wall-clock rate")
        self.ticks_per_ms = float(khz.value)
        self._next = 0

    def event(self) -> "ClockEvent":
        if self._next >= self.buf.numel():
            raise RuntimeError(f"device clock has only {self.buf.numel()} slots")
        self._next += 1
        return ClockEvent(self, self._next - 1)

    def refresh(self) -> None:
        self.host = self.buf.cpu().tolist()


class ClockEvent:
    """One timestamp slot of a :class:`DeviceClock`, with the ``record`` / ``elapsed_time`` of an event."""

    __slots__ = ("clock", "index")

    def __init__(self, clock: DeviceClock, index: int) -> None:
        self.clock, self.index = clock, index

    def record(self, stream: "HipStream | None" = None) -> "ClockEvent":
        s = stream if stream is not None else current_stream()
        nat.call("ftx_timestamp", self.clock.buf.data_ptr() + 8 * self.index, s.handle)
        return self

    def elapsed_time(self, end: "ClockEvent") -> float:
        h = self.clock.host
        return (h[end.index] - h[self.index]) / self.clock.ticks_per_ms


class HipStream:
    """A HIP stream. ``torch_stream`` keeps the owning torch object alive."""

    __slots__ = ("handle", "torch_stream", "name", "__weakref__")

    def __init__(self, torch_stream: Any = None, handle: int | None = None, name: str = "") -> None:
        self.torch_stream = torch_stream
        self.handle = int(handle if handle is not None else torch_stream.cuda_stream)
        self.name = name

    def record_event(self, event: HipEvent | None = None) -> HipEvent:
        return (event if event is not None else HipEvent()).record(self)

    def wait_event(self, event: HipEvent) -> None:
        nat.call("ftx_stream_wait_event", self.handle, event.handle)

    def wait_stream(self, other: "HipStream") -> None:
        self.wait_event(other.record_event())

    def synchronize(self) -> None:
        nat.call("ftx_stream_synchronize", self.handle)

    def query(self) -> bool:
        done = ctypes.c_int(0)
        nat.call("ftx_stream_query", self.handle, ctypes.byref(done))
        return bool(done.value)

    def __eq__(self, other: object) -> bool:
        return isinstance(other, HipStream) and other.handle == self.handle

    def __hash__(self) -> int:
        return hash(self.handle)

    def __repr__(self) -> str:
        return f"HipStream({self.name or hex(self.handle)})"


def is_capturing() -> bool:
    """Whether torch's current stream is capturing a graph (False without a GPU)."""
    return torch.cuda.is_available() and torch.cuda.is_current_stream_capturing()


def current_stream(device: torch.device | int | None = None) -> HipStream:
    """torch's current stream on ``device`` as a :class:`HipStream`."""
    return HipStream(torch.cuda.current_stream(device), name="compute")


def new_stream(device: torch.device | int | None = None, name: str = "transfer") -> HipStream:
    """A new stream at default priority, owned by torch's stream pool."""
    return HipStream(torch.cuda.Stream(device=device), name=name)


_TRANSFER_STREAMS: dict[int, HipStream] = {}
_REJECTED_STREAMS: list[Any] = []  # kept alive so later streams are not handed the same queue again
_STREAM_PROBES: dict[int, dict[str, Any]] = {}


class TransferStreamError(RuntimeError):
    """No new stream ran beside the compute stream: transfers would queue behind every forward kernel."""


def _probe_concurrency(candidate: HipStream, compute: HipStream, device: torch.device) -> tuple[float, float]:
    """``(busy_ms, candidate_ms)``: how long the compute stream's queued work took, and when a tiny fill
    queued on ``candidate`` at the same time finished.

    Streams share the device's hardware queues; a stream on the compute
    stream's queue waits behind every compute packet. The probe queues about
    two milliseconds of matrix products on ``compute`` (enqueued in a tenth of
    that) and a one-kilobyte fill on ``candidate``.
    """
    a = torch.ones(4096, 4096, dtype=torch.bfloat16, device=device)
    small = torch.empty(1024, dtype=torch.uint8, device=device)
    with torch.cuda.stream(compute.torch_stream) if compute.torch_stream is not None else _nullctx():
        torch.matmul(a, a)  # the first product at a shape selects its kernel on the host: keep that out of the window
    torch.cuda.synchronize(device)
    c_end, s_end, start = HipEvent(timing=True), HipEvent(timing=True), HipEvent(timing=True)
    compute.record_event(start)
    with torch.cuda.stream(compute.torch_stream) if compute.torch_stream is not None else _nullctx():
        for _ in range(16):
            torch.matmul(a, a)
    compute.record_event(c_end)
    with torch.cuda.stream(candidate.torch_stream):
        small.fill_(1)
    candidate.record_event(s_end)
    torch.cuda.synchronize(device)
    return start.elapsed_time(c_end), start.elapsed_time(s_end)


# A candidate on the compute stream's hardware queue finishes its fill only after all of the queued
# products (at about 100% of the busy time); one on another queue finishes within the first half, or
# around 60% when a profiler's tracing slows every dispatch. 80% separates the two.
_CONCURRENT_FRACTION = 0.8


def _runs_concurrently(candidate: HipStream, compute: HipStream, device: torch.device) -> bool:
    """Whether work on ``candidate`` finishes while ``compute`` is still busy."""
    busy, cand = _probe_concurrency(candidate, compute, device)
    return cand < _CONCURRENT_FRACTION * busy


def transfer_stream(device: torch.device | int | None = None, attempts: int = 8) -> HipStream:
    """The per-device stream used for host-to-device transfers.

    Chosen once per device among new default-priority streams: the first one
    whose work runs concurrently with torch's current stream (see
    :func:`_probe_concurrency`). Rejected candidates stay allocated, so the
    pool does not hand their queue out again. If none of ``attempts``
    candidates runs beside the compute stream, :class:`TransferStreamError`
    names the measurements. :func:`transfer_stream_probe` reports the outcome.
    """
    dev = torch.device("cuda", torch.cuda.current_device()) if device is None else torch.device(device)
    if dev.index is None:
        dev = torch.device("cuda", torch.cuda.current_device())
    cached = _TRANSFER_STREAMS.get(dev.index)
    if cached is not None:
        return cached
    compute = current_stream(dev)
    tried: list[tuple[float, float]] = []
    for i in range(attempts):
        cand = new_stream(dev, name="transfer")
        busy, done = _probe_concurrency(cand, compute, dev)
        tried.append((round(busy, 3), round(done, 3)))
        if done < _CONCURRENT_FRACTION * busy:
            _STREAM_PROBES[dev.index] = {"chosen_candidate": i, "rejected": i, "attempts": attempts,
                                         "compute_busy_ms": tried[-1][0], "transfer_fill_done_ms": tried[-1][1]}
            _TRANSFER_STREAMS[dev.index] = cand
            return cand
        _REJECTED_STREAMS.append(cand)
    raise TransferStreamError(
        f"no transfer stream on cuda:{dev.index} runs beside the compute stream: each of {attempts} new "
        f"default-priority streams finished a 1 KB fill only after the compute stream's queued matrix products "
        f"(compute busy ms, fill done ms per candidate: {tried}). Every candidate shares the compute stream's "
        "hardware queue, so transfers would wait behind each forward kernel; check GPU_MAX_HW_QUEUES and other "
        "work on this device")


def transfer_stream_probe(device: torch.device | int | None = None) -> dict[str, Any] | None:
    """How the transfer stream of ``device`` was chosen: candidate index, rejected count and the timings
    of the accepted probe; None before :func:`transfer_stream` ran there."""
    dev = torch.device("cuda", torch.cuda.current_device()) if device is None else torch.device(device)
    return _STREAM_PROBES.get(dev.index if dev.index is not None else torch.cuda.current_device())


@contextmanager
def use_stream(stream: HipStream) -> Iterator[None]:
    """Make ``stream`` torch's current stream inside the block."""
    if stream.torch_stream is None:
        raise ValueError("use_stream needs a stream created through torch")
    with torch.cuda.stream(stream.torch_stream):
        yield


class _ArenaOwner:
    """Frees one arena when the last reference to it goes away."""

    __slots__ = ("ptr",)

    def __init__(self, ptr: int) -> None:
        self.ptr = ptr

    def __del__(self) -> None:
        ptr, self.ptr = self.ptr, 0
        if not ptr:
            return
        try:
            if nat.live():
                nat.lib().ftx_arena_free(ptr)
        except (TypeError, AttributeError):
            pass  # interpreter shutdown: module globals are already gone; the process frees the arena


class HostArena:
    """Page-locked, device-mapped host bytes from ``ftx_arena_alloc``.

    ``tensor`` is a CPU ``uint8`` tensor over the arena. Ownership runs one
    way - tensor -> buffer -> owner - so the memory is returned by reference
    counting as soon as this object and every view of the tensor are gone
    (no cycle waits for the garbage collector while pinned memory is held).
    """

    def __init__(self, nbytes: int, flags: int = nat.ARENA_DEFAULT) -> None:
        if nbytes <= 0:
            raise ValueError(f"arena size must be positive, got {nbytes}")
        self.nbytes = int(nbytes)
        self.flags = flags
        self.ptr = nat.arena_alloc(self.nbytes, flags)
        owner = _ArenaOwner(self.ptr)
        self.device_ptr = nat.host_device_ptr(self.ptr)
        buf = (ctypes.c_uint8 * self.nbytes).from_address(self.ptr)
        buf._ftx_owner = owner  # every view holds the buffer, the buffer holds the owner
        self.tensor = torch.frombuffer(buf, dtype=torch.uint8)


def copy_h2d(dst: torch.Tensor, src: torch.Tensor, mode: int, stream: HipStream | None = None,
             nbytes: int | None = None, policy: nat.CopyPolicy | None = None) -> None:
    """Stream-ordered copy of ``nbytes`` (default: all of ``src``) host -> device, under ``policy`` (None: the
    library default)."""
    n = src.numel() * src.element_size() if nbytes is None else int(nbytes)
    if n > dst.numel() * dst.element_size():
        raise ValueError(f"copy of {n} bytes does not fit destination of {dst.numel() * dst.element_size()} bytes")
    if src.device.type != "cpu" or dst.device.type != "cuda":
        raise ValueError("copy_h2d needs a CPU source and a device destination")
    s = stream if stream is not None else current_stream(dst.device)
    nat.copy_h2d(dst.data_ptr(), src.data_ptr(), n, mode, s.handle, policy)


def checksum(t: torch.Tensor, stream: HipStream | None = None) -> int:
    """Device checksum of the bytes of a contiguous device tensor."""
    if t.device.type != "cuda" or not t.is_contiguous():
        raise ValueError("checksum needs a contiguous device tensor")
    s = stream if stream is not None else current_stream(t.device)
    return nat.checksum64(t.data_ptr(), t.numel() * t.element_size(), s.handle)


_PLAIN_TYPES = (torch.Tensor, torch.nn.Parameter)


def kernel_call(*tensors: torch.Tensor) -> bool:
    """Whether a call on these tensors may run a library kernel in place of torch operations: bf16 tensors on the
    current GPU, and nothing around the call that has to see torch operations - autograd, forward-mode
    differentiation, a function or dispatch mode (an offload manager's discovery is one), a functorch transform,
    autocast, or a trace."""
    first = tensors[0]
    if not first.is_cuda:
        return False
    c = torch._C
    if (torch.compiler.is_compiling() or c._get_tracing_state() is not None or c._len_torch_function_stack()
            or c._len_torch_dispatch_stack() or c._functorch.peek_interpreter_stack() is not None
            or torch.autograd.forward_ad._current_level >= 0 or torch.is_autocast_enabled("cuda")):
        return False
    grad = torch.is_grad_enabled()
    device = c._cuda_getDevice()
    bf16 = torch.bfloat16
    for t in tensors:
        if type(t) not in _PLAIN_TYPES or t.dtype != bf16 or t.get_device() != device or (grad and t.requires_grad):
            return False
    return True


def _packed(*tensors: torch.Tensor) -> bool:
    """Whether every tensor is contiguous and starts at a 16-byte boundary."""
    for t in tensors:
        if t.data_ptr() % 16 or not t.is_contiguous():
            return False
    return True


def _stream(device: int | None = None) -> int:
    """The handle of torch's current stream on ``device`` (None: the current device)."""
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice() if device is None else device)


def _head_strides(t: torch.Tensor) -> tuple[int, int, int] | None:
    """Batch, position and head strides of a [batch, position, head, d] tensor that can be read 16 bytes at a
    time, else None: contiguous along d, strides (of more than one element) multiples of 8, an aligned start."""
    s0, s1, s2, s3 = t.stride()
    n0, n1, n2, _ = t.shape
    s0, s1, s2 = s0 if n0 > 1 else 0, s1 if n1 > 1 else 0, s2 if n2 > 1 else 0
    return (s0, s1, s2) if s3 == 1 and not (s0 | s1 | s2) % 8 and t.data_ptr() % 16 == 0 else None


def _attention_sizes(b: int, t: int, s: int, h: int, kv: int, d: int, position_stride: int) -> bool:
    return (d in (64, 128) and b > 0 and t > 0 and s > 0 and kv > 0 and h > 0 and h % kv == 0
            and max(b, t * (h // kv), s) <= 1 << 24 and h <= 65536 and b * h * t <= 1 << 30
            and b * kv * ((t * (h // kv) + 31) // 32) < (1 << 26) - 64  # workgroups of one wave in one launch
            and (s + 256) * 2 * position_stride < 1 << 31)


def attention_eligible(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> bool:
    """Whether :func:`attention` takes these [batch, position, head, d] tensors."""
    if not kernel_call(q, k, v) or q.dim() != 4 or k.dim() != 4 or k.shape != v.shape:
        return False
    b, t, h, d = q.shape
    return (k.shape[0] == b and k.shape[3] == d
            and _attention_sizes(b, t, k.shape[1], h, k.shape[2], d, max(k.stride(1), v.stride(1)))
            and all(_head_strides(x) is not None for x in (q, k, v)))


_ATTENTION_WORKSPACE: dict[tuple, int] = {}


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, shape: tuple[int, ...], k_strides: tuple[int, ...],
            v_strides: tuple[int, ...], pos: int | None, stream: int) -> torch.Tensor:
    """The checked call: ``shape`` is (batch, queries, keys, heads, kv heads, d)."""
    out = torch.empty_like(q)
    ws_bytes = _ATTENTION_WORKSPACE.get(shape)
    if ws_bytes is None:
        got = ctypes.c_size_t(0)
        nat.call("ftx_attention_workspace", *shape, ctypes.byref(got))
        if len(_ATTENTION_WORKSPACE) >= 4096:  # a decode's key count grows by one a step
            _ATTENTION_WORKSPACE.clear()
        ws_bytes = _ATTENTION_WORKSPACE[shape] = int(got.value)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=q.device) if ws_bytes else None
    strides = (ctypes.c_int64 * 12)(*_head_strides(q), *k_strides, *v_strides, *_head_strides(out))
    nat.call("ftx_attention", q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), *shape, strides,
             0 if pos is None else 1, pos or 0, shape[5] ** -0.5, ws.data_ptr() if ws is not None else None, ws_bytes,
             stream)
    return out


def _check_operands(what: str, **tensors: torch.Tensor) -> None:
    """Refuses what a kernel must not read as plain bf16 memory of the current device, or would answer without
    the derivative that the caller asks for."""
    for name, t in tensors.items():
        if type(t) not in _PLAIN_TYPES:
            raise TypeError(f"{what} takes plain tensors, {name} is a {type(t).__name__}")
        if t.dtype != torch.bfloat16:
            raise TypeError(f"{what} takes bf16 tensors, {name} is {t.dtype}")
    for name, t in tensors.items():
        if not t.is_cuda or t.get_device() != torch._C._cuda_getDevice():
            raise ValueError(f"{what} runs on the current GPU, {name} is on {t.device}")
        if torch.is_grad_enabled() and t.requires_grad:
            raise ValueError(f"{what} has no backward and {name} requires a gradient")
        fwd = torch.autograd.forward_ad
        if fwd._current_level >= 0 and fwd.unpack_dual(t).tangent is not None:
            raise ValueError(f"{what} has no forward-mode derivative and {name} carries a tangent")


def attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, pos: int | None = None) -> torch.Tensor:
    """``softmax(q k^T / sqrt(d)) v`` over bf16 [batch, position, head, d] tensors (``ftx_attention``).

    ``k`` and ``v`` may have fewer heads than ``q`` (each shared by a group) and any strides; the result is laid
    out as q is. ``pos``: query t sees the keys up to ``pos + t``; None: every key. The tensors are on the current
    device, start at 16-byte boundaries and are contiguous along d, with strides that are multiples of 8; the
    kernel has no backward.
    """
    if not q.dim() == k.dim() == v.dim() == 4:
        raise ValueError(f"attention takes [batch, position, head, d] tensors, got {q.dim()}, {k.dim()} and {v.dim()} "
                         "dimensions")
    if k.shape != v.shape or k.shape[0] != q.shape[0] or k.shape[3] != q.shape[3]:
        raise ValueError(f"attention operands differ in batch, keys or head dimension: q {tuple(q.shape)}, "
                         f"k {tuple(k.shape)}, v {tuple(v.shape)}")
    _check_operands("attention", q=q, k=k, v=v)
    for name, t in (("q", q), ("k", k), ("v", v)):
        if _head_strides(t) is None:
            raise ValueError(f"attention reads {name} 16 bytes at a time: it must be contiguous along d and 16-byte "
                             f"aligned, with strides that are multiples of 8, not {t.stride()}")
    return attention_unchecked(q, k, v, pos)


def attention_unchecked(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, pos: int | None = None) -> torch.Tensor:
    """:func:`attention` for callers that have asked :func:`attention_eligible`."""
    b, t, h, d = q.shape
    return _attend(q, k, v, (b, t, k.shape[1], h, k.shape[2], d), _head_strides(k), _head_strides(v), pos, _stream())


NORM_MAX_DIM = 32768


def _norm_rows_fit(rows: int, dim: int) -> bool:
    """Whether one launch (fewer than 2^32 threads) holds these rows of 1, 4 or 16 waves."""
    return rows * (64 if dim <= 2048 else 256 if dim <= 8192 else 1024) <= (1 << 32) - 4096


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor | None:
    """``bf16(x * rsqrt(mean(x^2) + eps) * weight)`` over the last dimension in one launch (``ftx_norm``), or
    None when the kernel does not take the call."""
    if type(x) not in _PLAIN_TYPES:  # a subclass, or a proxy of a symbolic trace
        return None
    dim = x.shape[-1] if x.dim() else 0
    numel = x.numel()
    if (not dim or dim % 8 or dim > NORM_MAX_DIM or not numel
            or (numel > 1 << 28 and not _norm_rows_fit(numel // dim, dim))
            or not kernel_call(x, weight) or weight.shape != (dim,) or not _packed(x, weight)):
        return None
    y = torch.empty_like(x)
    nat.call("ftx_norm", x.data_ptr(), None, None, y.data_ptr(), numel // dim, dim, nat.NORM_RMS,
             weight.data_ptr(), None, None, None, 1, -1, -1, -1, eps, _stream())
    return y


def residual_norm(x: torch.Tensor, eps: float, delta: torch.Tensor | None = None, gate: int = -1,
                  affine: tuple[torch.Tensor, torch.Tensor] | None = None,
                  adaln: tuple[torch.Tensor, torch.Tensor] | None = None, scale: int = -1,
                  shift: int = -1) -> tuple[torch.Tensor, torch.Tensor | None] | None:
    """``(sum, normalised)`` of bf16 [batch, n, dim] rows in one launch (``ftx_norm``), or None when the kernel
    does not take the call.

    The sum is ``x``, ``x + delta``, or ``x + delta * m[gate]``; the normalised rows (None for none of the two)
    are its LayerNorm with ``affine`` (weight, bias), or ``LayerNorm(sum) * (1 + m[scale]) + m[shift]`` for a
    ``scale`` that is not negative. ``m = modulation + e`` from ``adaln``: [1, 6, dim] and [batch, 6, dim].
    """
    if type(x) not in _PLAIN_TYPES or x.dim() != 3 or not x.numel():
        return None
    b, n, dim = x.shape
    if affine is not None and (affine[0] is None or affine[1] is None):  # a LayerNorm without a weight or a bias
        return None
    tensors = [t for t in (x, delta, *(affine or ()), *(adaln or ())) if t is not None]
    if (dim % 8 or dim > NORM_MAX_DIM or not _norm_rows_fit(b * n, dim) or not kernel_call(*tensors)
            or not _packed(*tensors) or (delta is not None and delta.shape != x.shape)
            or (affine is not None and not affine[0].shape == affine[1].shape == (dim,))
            or (adaln is not None and (adaln[0].shape != (1, 6, dim) or adaln[1].shape != (b, 6, dim)))):
        return None
    norm = nat.NORM_ADALN if scale >= 0 else nat.NORM_LAYER if affine is not None else nat.NORM_NONE
    total = torch.empty_like(x) if delta is not None else x
    y = torch.empty_like(x) if norm != nat.NORM_NONE else None
    ptr = [t.data_ptr() if t is not None else None for t in (delta, total, y, *(affine or (None, None)),
                                                             *(adaln or (None, None)))]
    nat.call("ftx_norm", x.data_ptr(), ptr[0], ptr[1], ptr[2], b * n, dim, norm, ptr[3], ptr[4], ptr[5], ptr[6], n,
             gate, scale, shift, eps, _stream())
    return total, y


def _rope(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, pos: int,
          cache_k: torch.Tensor, cache_v: torch.Tensor, stream: int):
    """:func:`rope_cache`, with the caches' strides: ``(rotated q, cache_k strides, cache_v strides)``."""
    b, t, h, d = q.shape
    kv = k.shape[2]
    if (type(pos) is not int or pos < 0 or d % 16 or not 0 < b * t * (h + 2 * kv) * d <= 1 << 35 or not h
            or k.shape != (b, t, kv, d) or v.shape != k.shape or not _packed(q, k, v)):
        return None
    grad = torch.is_grad_enabled()
    device = q.get_device()
    for table in (cos, sin):
        if (type(table) not in _PLAIN_TYPES or table.dtype != torch.float32 or table.dim() != 2
                or table.shape[1] != d or table.shape[0] < pos + t or table.get_device() != device
                or (grad and table.requires_grad) or not _packed(table)):
            return None
    strides = []
    for cache in (cache_k, cache_v):
        if cache.dim() != 4 or cache.shape[0] < b or cache.shape[1] < pos + t or cache.shape[2:] != (kv, d):
            return None
        strides.append(_head_strides(cache))
        if (strides[-1] is None or 0 in cache.stride()
                or (cache.is_inference() and not torch.is_inference_mode_enabled())):
            return None
    if cache_k.data_ptr() == cache_v.data_ptr():
        return None
    torch._C._increment_version((cache_k, cache_v))  # as an in-place operation, for what autograd saved
    out = torch.empty_like(q)
    nat.call("ftx_rope_cache", q.data_ptr(), k.data_ptr(), v.data_ptr(), cos.data_ptr(), sin.data_ptr(),
             out.data_ptr(), cache_k.data_ptr(), cache_v.data_ptr(), b, t, h, kv, d, pos,
             (ctypes.c_int64 * 6)(*strides[0], *strides[1]), stream)
    return out, *strides


def rope_cache(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, pos: int,
               cache_k: torch.Tensor, cache_v: torch.Tensor) -> torch.Tensor | None:
    """The rotated queries of [batch, t, head, d] ``q``; the rotated ``k`` and ``v`` go to positions ``pos ..
    pos + t - 1`` of the caches, in one launch (``ftx_rope_cache``). None when the kernel does not take the
    call."""
    b, t, h, d = q.shape
    if max(b, t) > 1 << 24 or max(h, k.shape[2]) > 65536 or d > 4096 or not kernel_call(q, k, v, cache_k, cache_v) or (
            type(pos) is int and pos > 1 << 30):
        return None
    got = _rope(q, k, v, cos, sin, pos, cache_k, cache_v, _stream())
    return got[0] if got is not None else None


def rope_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, pos: int,
                   cache_k: torch.Tensor, cache_v: torch.Tensor) -> torch.Tensor | None:
    """Causal attention of new positions over the KV cache: :func:`rope_cache`, then :func:`attention` of the
    rotated queries over the first ``pos + t`` cached positions. None, with nothing written, when the kernels do
    not take the call."""
    if type(pos) is not int:
        return None
    b, t, h, d = q.shape
    shape = (b, t, pos + t, h, k.shape[2], d)
    if (not kernel_call(q, k, v, cache_k, cache_v) or cache_k.dim() != 4 or cache_v.dim() != 4
            or not _attention_sizes(*shape, max(cache_k.stride(1), cache_v.stride(1)))):
        return None
    stream = _stream()
    got = _rope(q, k, v, cos, sin, pos, cache_k, cache_v, stream)
    return _attend(got[0], cache_k, cache_v, shape, got[1], got[2], pos, stream) if got is not None else None


def silu_mul(g: torch.Tensor, u: torch.Tensor) -> torch.Tensor | None:
    """``bf16(bf16(silu(g)) * u)`` in one launch (``ftx_silu_mul``), or None when the kernel does not take the
    call."""
    n = g.numel()
    if g.shape != u.shape or not n or n % 8 or n > (1 << 35) - 4096 or not kernel_call(g, u) or not _packed(g, u):
        return None
    y = torch.empty_like(g)
    nat.call("ftx_silu_mul", g.data_ptr(), u.data_ptr(), y.data_ptr(), n, _stream())
    return y


FP8_DECODE_MAX_ROWS = 64  # more rows run the tiled prefill kernel
_FP8_WORKSPACE: dict[tuple, int] = {}


def fp8_linear_workspace_bytes(m: int, n: int, k: int) -> int:
    """Bytes of device workspace one ``fp8_linear`` call of this shape needs (cached per shape)."""
    key = (m, n, k)
    got = _FP8_WORKSPACE.get(key)
    if got is None:
        b = ctypes.c_size_t(0)
        nat.call("ftx_fp8_linear_workspace", m, n, k, ctypes.byref(b))
        got = _FP8_WORKSPACE[key] = int(b.value)
    return got


def fp8_linear_scratch_bytes(m: int, ns: tuple[int, ...], k: int, epilogue: int = nat.FP8_EPILOGUE_NONE) -> int:
    """Bytes of workspace a call touches under the launch shape in force, 0 for one launch (cached per shape)."""
    key = ("scratch", epilogue, m, k) + ns
    got = _FP8_WORKSPACE.get(key)
    if got is None:
        b = ctypes.c_size_t(0)
        nat.call("ftx_fp8_linear_scratch", m, (ctypes.c_int64 * len(ns))(*ns), len(ns), k, epilogue, ctypes.byref(b))
        got = _FP8_WORKSPACE[key] = int(b.value)
    return got


def _check_fp8_operands(what: str, x: torch.Tensor, weight: torch.Tensor, scale: torch.Tensor) -> tuple[int, int, int]:
    """Ranks, dtypes, shapes and devices of an fp8 linear's operands; returns (m, k, n)."""
    if x.dim() != 2 or weight.dim() != 2 or scale.dim() != 1:
        raise ValueError(f"{what} needs x [m, k], weight [n, k] and scale [n]")
    if x.dtype != torch.bfloat16 or weight.dtype != torch.float8_e4m3fn or scale.dtype != torch.bfloat16:
        raise TypeError(f"{what} needs bf16 x, float8_e4m3fn weight and bf16 scale; got "
                        f"{x.dtype}, {weight.dtype}, {scale.dtype}")
    m, k = x.shape
    n = weight.shape[0]
    if weight.shape[1] != k or scale.shape[0] != n:
        raise ValueError(f"shape mismatch: x {tuple(x.shape)}, weight {tuple(weight.shape)}, scale {tuple(scale.shape)}")
    if not (x.is_cuda and weight.device == x.device and scale.device == x.device):
        raise ValueError(f"{what} needs x, weight and scale on one GPU")
    return m, k, n


def fp8_linear(x: torch.Tensor, weight: torch.Tensor, scale: torch.Tensor) -> torch.Tensor:
    """``bf16(scale * (x @ weight.T))`` by the library's fp8-weight MFMA kernel.

    ``x``: bf16 ``[m, k]``; ``weight``: float8 e4m3fn ``[n, k]``; ``scale``:
    bf16 ``[n]``; all on one device. The weights are widened to bf16 in
    registers, so the products are those of dequantizing and running a bf16
    GEMM. A few rows run in one launch, up to 64 the split-K decode kernel,
    more rows the tiled prefill kernel. Runs on torch's current stream; a
    split-K workspace comes from torch's allocator on that stream.
    """
    m, k, n = _check_fp8_operands("fp8_linear", x, weight, scale)
    if not weight.is_contiguous() or weight.data_ptr() % 16:
        raise ValueError("fp8_linear needs a contiguous, 16-byte aligned weight")
    if not x.is_contiguous() or x.data_ptr() % 16:
        x = x.clone(memory_format=torch.contiguous_format)
    if not scale.is_contiguous():
        scale = scale.contiguous()
    y = torch.empty((m, n), dtype=torch.bfloat16, device=x.device)
    ws_bytes = fp8_linear_scratch_bytes(m, (n,), k, nat.FP8_EPILOGUE_NONE)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=x.device) if ws_bytes else None
    nat.call("ftx_fp8_linear", x.data_ptr(), weight.data_ptr(), scale.data_ptr(), y.data_ptr(), m, n, k,
             ws.data_ptr() if ws is not None else None, ws_bytes, _stream(x.get_device()))
    return y


def fp8_linear_group_workspace_bytes(m: int, ns: list[int], k: int) -> int:
    """Bytes of device workspace one ``fp8_linear_group`` call of these shapes needs (cached per shape)."""
    key = ("group", m, k) + tuple(ns)  # distinct from the (m, n, k) keys of single calls
    got = _FP8_WORKSPACE.get(key)
    if got is None:
        arr = (ctypes.c_int64 * len(ns))(*ns)
        b = ctypes.c_size_t(0)
        nat.call("ftx_fp8_linear_group_workspace", m, ctypes.cast(arr, ctypes.c_void_p), len(ns), k, ctypes.byref(b))
        got = _FP8_WORKSPACE[key] = int(b.value)
    return got


def fp8_linear_group(x: torch.Tensor, weights: list[torch.Tensor], scales: list[torch.Tensor]) -> list[torch.Tensor]:
    """``[fp8_linear(x, w, s) for w, s in zip(weights, scales)]`` in one launch (``ftx_fp8_linear_group``).

    For up to four weight matrices that share ``x`` and ``k`` (a layer's q/k/v or gate/up projections): the
    group pays one kernel launch, and one reduce launch when K is split, instead of one of each per matrix.
    Each output equals the single call's to within fp32 rounding (the group may split K differently).
    """
    if not 1 <= len(weights) <= 4 or len(weights) != len(scales):
        raise ValueError("fp8_linear_group takes 1 to 4 weights with one scale each")
    if x.dim() != 2 or x.dtype != torch.bfloat16 or not x.is_cuda:
        raise ValueError("fp8_linear_group needs a bf16 GPU x [m, k]")
    m, k = x.shape
    for w, sc in zip(weights, scales):
        if w.dtype != torch.float8_e4m3fn or w.dim() != 2 or w.shape[1] != k or w.device != x.device:
            raise ValueError(f"every weight must be float8_e4m3fn [n, {k}] on {x.device}")
        if not w.is_contiguous() or w.data_ptr() % 16:
            raise ValueError("fp8_linear_group needs contiguous, 16-byte aligned weights")
        if sc.dtype != torch.bfloat16 or sc.shape != (w.shape[0],) or sc.device != x.device:
            raise ValueError("every scale must be bf16 [n] on the input's device")
    if not x.is_contiguous() or x.data_ptr() % 16:
        x = x.clone(memory_format=torch.contiguous_format)
    scales = [sc if sc.is_contiguous() else sc.contiguous() for sc in scales]
    g = len(weights)
    ns = (ctypes.c_int64 * g)(*[w.shape[0] for w in weights])
    outs = [torch.empty((m, w.shape[0]), dtype=torch.bfloat16, device=x.device) for w in weights]
    ws_bytes = fp8_linear_scratch_bytes(m, tuple(ns), k, nat.FP8_EPILOGUE_NONE)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=x.device) if ws_bytes else None
    ptrs = [(ctypes.c_void_p * g)(*[t.data_ptr() for t in ts]) for ts in (weights, scales, outs)]
    nat.call("ftx_fp8_linear_group", x.data_ptr(), g, *ptrs, ns, m, k, ws.data_ptr() if ws is not None else None,
             ws_bytes, _stream(x.get_device()))
    return outs


def fp8_linear_fused_workspace_bytes(m: int, ns: list[int], k: int, epilogue: int) -> int:
    """Bytes of device workspace one ``ftx_fp8_linear_fused`` call of these shapes needs (cached per shape)."""
    key = ("fused", epilogue, m, k) + tuple(ns)
    got = _FP8_WORKSPACE.get(key)
    if got is None:
        arr = (ctypes.c_int64 * len(ns))(*ns)
        b = ctypes.c_size_t(0)
        nat.call("ftx_fp8_linear_fused_workspace", m, ctypes.cast(arr, ctypes.c_void_p), len(ns), k, epilogue,
                 ctypes.byref(b))
        got = _FP8_WORKSPACE[key] = int(b.value)
    return got


def _fp8_fused(x: torch.Tensor, weights: list[torch.Tensor], scales: list[torch.Tensor], epilogue: int,
               residual: torch.Tensor | None, what: str) -> torch.Tensor:
    ms = [_check_fp8_operands(what, x, w, sc) for w, sc in zip(weights, scales)]
    m, k, n = ms[0]
    if m > FP8_DECODE_MAX_ROWS:
        raise ValueError(f"{what} runs in the decode kernel: at most {FP8_DECODE_MAX_ROWS} rows, got {m}")
    for w in weights:
        if not w.is_contiguous() or w.data_ptr() % 16:
            raise ValueError(f"{what} needs contiguous, 16-byte aligned weights")
    if not x.is_contiguous() or x.data_ptr() % 16:
        x = x.clone(memory_format=torch.contiguous_format)
    scales = [sc if sc.is_contiguous() else sc.contiguous() for sc in scales]
    if residual is not None:
        if residual.shape != (m, n) or residual.dtype != torch.bfloat16 or residual.device != x.device:
            raise ValueError(f"{what}: the residual must be bf16 [{m}, {n}] on {x.device}")
        if not residual.is_contiguous():
            residual = residual.contiguous()
    g = len(weights)
    ns = [w.shape[0] for w in weights]
    y = torch.empty((m, n), dtype=torch.bfloat16, device=x.device)
    ws_bytes = fp8_linear_scratch_bytes(m, tuple(ns), k, epilogue)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=x.device) if ws_bytes else None
    arrays = [(ctypes.c_void_p * g)(*[t.data_ptr() for t in ts]) for ts in (weights, scales)]
    n_arr = (ctypes.c_int64 * g)(*ns)
    nat.call("ftx_fp8_linear_fused", x.data_ptr(), g, *arrays, y.data_ptr(), n_arr, m, k, epilogue,
             residual.data_ptr() if residual is not None else None, ws.data_ptr() if ws is not None else None, ws_bytes,
             _stream(x.get_device()))
    return y


def fp8_linear_swiglu(x: torch.Tensor, w_gate: torch.Tensor, s_gate: torch.Tensor, w_up: torch.Tensor,
                      s_up: torch.Tensor) -> torch.Tensor:
    """``F.silu(g) * u`` for ``g, u = fp8_linear(x, w_gate, s_gate), fp8_linear(x, w_up, s_up)`` in one grouped
    launch plus its reduce (``FTX_FP8_EPILOGUE_SWIGLU``): a SwiGLU MLP's gate and up projections and their
    activation. Decode batches only (at most 64 rows); g and u are rounded to bf16 as the separate
    projections round them, silu(g) is rounded to bf16, then the product."""
    if w_gate.shape != w_up.shape:
        raise ValueError(f"gate and up weights differ in shape: {tuple(w_gate.shape)} and {tuple(w_up.shape)}")
    return _fp8_fused(x, [w_gate, w_up], [s_gate, s_up], nat.FP8_EPILOGUE_SWIGLU, None, "fp8_linear_swiglu")


def fp8_linear_residual(x: torch.Tensor, weight: torch.Tensor, scale: torch.Tensor,
                        residual: torch.Tensor) -> torch.Tensor:
    """``residual + fp8_linear(x, weight, scale)`` with the add folded into the reduce
    (``FTX_FP8_EPILOGUE_RESIDUAL``): a decoder's output projection and its residual connection. Decode
    batches only (at most 64 rows); the same bits as the separate linear and bf16 add."""
    return _fp8_fused(x, [weight], [scale], nat.FP8_EPILOGUE_RESIDUAL, residual, "fp8_linear_residual")


BF16_LINEAR_MAX_ROWS = 16


def _bf16_linear_wins(m: int, n: int, k: int) -> bool:
    """Whether the one-launch kernel is faster than the library's GEMM for ``m`` rows of one [n, k] weight.

    It is at every n from K = 2048 on (1.05 times its time at worst, 131072 x 3072 at 16 rows). Of a shorter K each
    workgroup has little to do for its 16 channels, so many of them lose. Its time by the library's at 4, 8 and 16
    rows: 8192 x 64 0.76, 0.79, 0.91 and 32768 x 64 1.65, 1.82, 1.94; 16384 x 256 0.81, 0.89, 1.03 and 65536 x 256
    1.49, 1.59, 1.80; 32768 x 512 0.81, 0.88, 0.97 and 65536 x 512 1.12, 1.19, 1.35; 65536 x 1024 0.92, 1.05, 1.28.
    The choice looks at one weight, so a projection has the same bits alone and in a group.
    """
    return n <= 8192 or k >= 2048 or (m <= 8 and k >= 1536) or n <= (64 if m <= 4 else 48 if m <= 8 else 12) * k


def bf16_linear_eligible(x: torch.Tensor, *weights: torch.Tensor) -> bool:
    """Whether ``x`` [..., k] and these weights [n, k] are better off in :func:`bf16_linear` than in torch's linear,
    and may run there."""
    if type(x) not in _PLAIN_TYPES:  # a subclass, or a proxy of a symbolic trace
        return False
    k = x.shape[-1] if x.dim() else 0
    numel = x.numel()
    if not 0 < k <= 1 << 29 or not 0 < numel <= BF16_LINEAR_MAX_ROWS * k or k % 8 or not kernel_call(x, *weights):
        return False
    channels = 0
    for w in weights:
        shape = w.shape
        n = shape[0] if len(shape) == 2 and shape[1] == k else 0
        if not n or (k < 2048 and not _bf16_linear_wins(numel // k, n, k)):
            return False
        channels += n
    return channels <= (1 << 27) - 128 and _packed(x, *weights)  # channels of one launch


def bf16_linear(x: torch.Tensor, weights: list[torch.Tensor], epilogue: int = nat.FP8_EPILOGUE_NONE,
                residual: torch.Tensor | None = None) -> list[torch.Tensor]:
    """``[x @ w.T for w in weights]`` for up to 16 bf16 rows in one launch (``ftx_bf16_linear``); under an
    epilogue one output: ``silu(g) * u`` of two weights, or ``residual + x @ w.T`` of one. ``x`` [..., k] and the
    weights [n, k] are contiguous, 16-byte aligned and on the current device; the kernel has no backward."""
    k = x.shape[-1] if x.dim() else 0
    if k == 0:
        raise ValueError(f"bf16_linear takes x [..., k], got {tuple(x.shape)}")
    named = {"x": x, **{f"weights[{i}]": w for i, w in enumerate(weights)}}
    for name, t in named.items():
        if t is not x and (t.dim() != 2 or t.shape[1] != k):
            raise ValueError(f"bf16_linear: {name} must be [n, {k}], got {tuple(t.shape)}")
        if not _packed(t):
            raise ValueError(f"bf16_linear needs a contiguous, 16-byte aligned {name}")
    if epilogue == nat.FP8_EPILOGUE_RESIDUAL and residual is not None and weights:
        shape = (*x.shape[:-1], weights[0].shape[0])
        if residual.shape != shape or not residual.is_contiguous():
            raise ValueError(f"residual must be a contiguous {shape} tensor, got {tuple(residual.shape)}")
        named["residual"] = residual
    _check_operands("bf16_linear", **named)
    return bf16_linear_unchecked(x, weights, epilogue, residual)


def bf16_linear_unchecked(x: torch.Tensor, weights: list[torch.Tensor], epilogue: int = nat.FP8_EPILOGUE_NONE,
                          residual: torch.Tensor | None = None) -> list[torch.Tensor]:
    """:func:`bf16_linear` for callers that have asked :func:`bf16_linear_eligible`."""
    k = x.shape[-1]
    m, g = x.numel() // k, len(weights)
    n_out = 1 if epilogue == nat.FP8_EPILOGUE_SWIGLU else g
    outs = [torch.empty((*x.shape[:-1], w.shape[0]), dtype=torch.bfloat16, device=x.device) for w in weights[:n_out]]
    ptrs = ctypes.c_void_p * g
    nat.call("ftx_bf16_linear", x.data_ptr(), g, ptrs(*[w.data_ptr() for w in weights]),
             ptrs(*[y.data_ptr() for y in outs]), (ctypes.c_int64 * g)(*[w.shape[0] for w in weights]), m, k, epilogue,
             residual.data_ptr() if residual is not None else None, _stream())
    return outs


def fp8_linear_static(x: torch.Tensor, weight: torch.Tensor, scale: torch.Tensor, out: torch.Tensor) -> torch.Tensor:
    """``fp8_linear`` into ``out`` (bf16 ``[m, n]``) with no allocation at all, for graph capture and serving
    loops: the split-K partial sums live in the library's static per-GPU scratch array
    (``ftx_fp8_linear_static``). Operands must already be contiguous and 16-byte aligned. Calls that may
    overlap on one GPU share that scratch and must be ordered (one stream). Every operand is checked as
    ``fp8_linear`` checks it (dtypes, shapes, one device); nothing is copied to fix a layout."""
    m, k, n = _check_fp8_operands("fp8_linear_static", x, weight, scale)
    if out.shape != (m, n) or out.dtype != torch.bfloat16 or not out.is_contiguous() or out.device != x.device:
        raise ValueError(f"out must be a contiguous bf16 [{m}, {n}] tensor on {x.device}")
    for name, t in (("x", x), ("weight", weight)):
        if not t.is_contiguous() or t.data_ptr() % 16:
            raise ValueError(f"fp8_linear_static needs a contiguous, 16-byte aligned {name}")
    if not scale.is_contiguous():
        raise ValueError("fp8_linear_static needs a contiguous scale")
    nat.call("ftx_fp8_linear_static", x.data_ptr(), weight.data_ptr(), scale.data_ptr(), out.data_ptr(), m, n, k,
             torch.cuda.current_stream(x.device).cuda_stream)
    return out


def set_fp8_linear_config(waves: int = 0, slice_k: int = 0) -> None:
    """Fix the fp8 linear launch shape: wavefronts per workgroup and K values
    per workgroup (0 = chosen per call from the shape)."""
    nat.call("ftx_set_fp8_linear_config", waves, slice_k)
    _FP8_WORKSPACE.clear()
