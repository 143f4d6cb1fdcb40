"""Small helpers shared by the host-side wrappers (device checks, streams, dtypes)."""
from __future__ import annotations

import functools
import threading

import torch

from . import _lib

_DTYPE_CODE = {torch.bfloat16: _lib.DTYPE_BF16, torch.float16: _lib.DTYPE_FP16,
               torch.float32: _lib.DTYPE_FP32}


def dtype_code(dt: torch.dtype, allowed=(torch.bfloat16, torch.float16, torch.float32)) -> int:
    if dt not in allowed:
        raise ValueError(f"unsupported dtype {dt}; expected one of {allowed}")
    return _DTYPE_CODE[dt]


def require_gpu(what: str, *tensors) -> torch.device:
    """All tensors must live on one ROCm GPU: this package has no CPU path."""
    dev = None
    for t in tensors:
        if t is None:
            continue
        if not isinstance(t, torch.Tensor) or not t.is_cuda:
            raise ValueError(f"{what}: expected tensors on a ROCm GPU device, got "
                             f"{getattr(t, 'device', type(t))}; batchspec_amd has no CPU path")
        d = t.device
        if dev is None:
            dev = d
        elif d != dev:
            raise ValueError(f"{what}: tensors on different devices ({dev} and {d})")
    if dev is None:
        raise ValueError(f"{what}: no tensor given")
    return dev


# torch's current raw stream of a device index.  torch.cuda.current_stream() builds a Stream
# object around the same address, about 2 us of a 15-20 us call.
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def stream_of(device: torch.device) -> int:
    """hipStream_t of torch's current stream on `device` (as an integer address)."""
    if _raw_stream is None:
        return torch.cuda.current_stream(device).cuda_stream
    index = device.index
    return _raw_stream(torch.cuda.current_device() if index is None else index)


@functools.lru_cache(maxsize=None)
def num_cus(device_index: int) -> int:
    return torch.cuda.get_device_properties(device_index).multi_processor_count


# Held from a call's choice of a workspace until its launches are queued: the launches of
# one call share the workspace, so two host threads on one stream must not interleave theirs
# (ctypes releases the GIL during the call).
LAUNCH_LOCK = threading.Lock()


_MAX_WORKSPACES = 64  # eager ones of a cache: torch has 32 pooled streams


def workspace(device: torch.device, nbytes: int, cache: dict, name: str,
              stream: int) -> torch.Tensor:
    """A uint8 device buffer of at least `nbytes`, reused through `cache` by the calls of
    `name` on this device and stream, which must be the current one (the caller holds
    LAUNCH_LOCK).

    One per stream: a call's kernels hand results to each other through it, and calls on
    different streams may run at the same time.  Dropping one is safe: the allocator gives
    its memory only to later work on the same stream.
    Captured calls take buffers of their own, since a graph may replay beside eager work on
    any stream, and those are never freed ("__retired__"): the graph holds their addresses
    as kernel arguments.  Growth doubles, so the outgrown ones stay below the current one.
    Graphs captured on one stream share a buffer: their replays must not overlap."""
    nbytes = max(int(nbytes), 256)
    captured = torch.cuda.is_current_stream_capturing()
    key = (name, device.index, stream, captured)
    buf = cache.get(key)
    if buf is not None and buf.numel() >= nbytes:
        return buf
    if buf is not None:
        nbytes = max(nbytes, 2 * buf.numel())
    buf = torch.empty(nbytes, dtype=torch.uint8, device=device)
    if captured:
        cache.setdefault("__retired__", []).append(buf)
    else:
        eager = [k for k in cache if k != "__retired__" and not k[3] and k != key]
        if len(eager) >= _MAX_WORKSPACES:
            del cache[eager[0]]
    cache[key] = buf
    return buf
