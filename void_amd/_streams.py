"""The current HIP stream, and arrays used on several."""

from __future__ import annotations

import torch


def raw_stream(device: torch.device) -> int:
    """Handle of torch's current stream on a GPU device
    (torch.cuda.current_stream(device).cuda_stream without the Stream object)."""
    return torch._C._cuda_getCurrentRawStream(device.index if device.index is not None
                                              else torch.cuda.current_device())


def record_once(seen: set, device: torch.device, *arrays: torch.Tensor) -> None:
    """Record GPU arrays on the current stream, once for each stream (seen: the
    raw streams so far).  The allocator then gives their memory out again only
    when what was queued on these streams before they were freed is done; a
    caller between this and its launch still holds them, so its launch is
    queued before.  (record_stream lasts until the array is freed.)"""
    raw = raw_stream(device)
    if raw not in seen:
        for t in arrays:
            t.record_stream(torch.cuda.current_stream(device))
        seen.add(raw)
