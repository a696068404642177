"""Device plumbing for driving the gfx950 packs from Python.

PyTorch is used only for device memory and streams.  Every entry point of
the packs rejects stream 0 (the reference's "explicit engine stream" rule,
src/backend/cuda/gemm_plan.cpp:181-184), so callers run under
``engine_stream()``, which makes a dedicated (default-priority) HIP stream
current for both torch allocations and pack launches.
"""
from __future__ import annotations

import contextlib
from typing import Optional

import torch

_stream: Optional["torch.cuda.Stream"] = None


def require_gpu() -> None:
    if not torch.cuda.is_available():
        raise RuntimeError("pih_amd: no HIP device visible; the gfx950 packs have no CPU fallback")


def stream() -> "torch.cuda.Stream":
    global _stream
    if _stream is None:
        require_gpu()
        _stream = torch.cuda.Stream()
    return _stream


class engine_stream(contextlib.ContextDecorator):
    """``with engine_stream() as s``: the engine stream is torch's current
    stream inside.  The same switch as ``torch.cuda.stream(s)``; entering and
    leaving through the two calls that one ends in took 7.6 -> 1.6 us, of the
    ~27 us of host time around a four-launch decode block.

    A context object is entered once, as a generator's is: what to go back to
    is kept on it, so that entered again, or by a second thread, it would
    leave the engine stream current.  Call ``engine_stream()`` for each."""

    def __init__(self) -> None:
        self._unused = [True]

    def _recreate_cm(self):  # as a decorator: a context of its own per call
        return engine_stream()

    def __enter__(self):
        try:
            self._unused.pop()  # one thread gets it
        except IndexError:
            raise RuntimeError("pih_amd: an engine_stream() context is entered once") from None
        s = stream()
        self._other = None
        if torch._C._cuda_getDevice() != s.device_index:
            # another device is current: torch's own context restores both
            self._other = torch.cuda.stream(s)
            self._other.__enter__()
        else:
            self._previous = torch._C._cuda_getCurrentStream(s.device_index)
            torch._C._cuda_setStream(stream_id=s.stream_id, device_index=s.device_index, device_type=s.device_type)
        return s

    def __exit__(self, *exc):
        if self._other is not None:
            self._other.__exit__(*exc)
        else:
            sid, index, kind = self._previous
            torch._C._cuda_setStream(stream_id=sid, device_index=index, device_type=kind)
        return False


def stream_handle() -> int:
    # the current stream's handle without a Stream object (2.8 -> 0.3 us)
    h = torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())
    if h == 0:
        raise RuntimeError("pih_amd: launches need an explicit stream; run under pih_amd.device.engine_stream()")
    return h


def ptr(t: Optional[torch.Tensor]) -> int:
    if t is None:
        return 0
    if not t.is_cuda:
        raise ValueError("pih_amd: tensor must live on the HIP device")
    if not t.is_contiguous():
        raise ValueError("pih_amd: tensor must be contiguous")
    return t.data_ptr()


def error_flag() -> torch.Tensor:
    return torch.zeros(1, dtype=torch.int32, device="cuda")


def flag_value(flag: torch.Tensor) -> int:
    return int(flag.item()) & 0xFFFFFFFF
