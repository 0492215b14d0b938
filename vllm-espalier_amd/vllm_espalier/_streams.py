"""Buffers kept across calls, and the streams that use them."""
import torch

_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)      # None: a torch without a GPU


def raw_stream(device):
    """The handle of the device's current stream; None for the CPU."""
    if device.type != "cuda":
        return None
    return _raw_stream(torch.cuda.current_device() if device.index is None else device.index)


def hand_out(tensors, seen: set, device, raw) -> None:
    """Tell the caching allocator that `tensors`, kept across calls and dropped once outgrown, are used on the device's current
    stream too (raw_stream's, not yet in `seen`, the streams already told; once is enough for a tensor's life). Freed memory
    goes back to the stream that allocated it, which need not wait for another stream's launches; from here on the allocator
    holds it until this stream has run what it was given by then. Not for a capture, whose buffers the caller keeps."""
    stream = torch.cuda.current_stream(device)
    for t in tensors:
        t.record_stream(stream)              # nothing to tell on the stream that allocated it
    seen.add(raw)
