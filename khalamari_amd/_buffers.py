"""Borrowed device buffers for the C ABI: anything with `data_ptr()` (a torch tensor) or a (ptr, bytes) pair."""
from __future__ import annotations

from array import array
from ctypes import sizeof

from ._lib import Buffer

NO_BUFFER = Buffer(None, 0)


def view(obj) -> Buffer:
    if isinstance(obj, Buffer):
        return obj
    if isinstance(obj, tuple):
        return Buffer(int(obj[0]), int(obj[1]))
    if hasattr(obj, "data_ptr"):
        return Buffer(obj.data_ptr(), obj.numel() * obj.element_size())
    raise TypeError(f"cannot borrow {type(obj).__name__} as a device buffer")


def pack(struct_type, *objects):
    """A structure whose fields are all `Buffer`s from what `view` accepts, in field order.  A decode step of one request is
    two launches of a few microseconds each, and a ctypes structure per buffer took longer than they do: the (pointer, length)
    words go into one array that the structure is laid over (a call with thirteen buffers and three counts 14.6 -> 8.3 us, the
    projection prologue with its configs 13.5 -> 6.4 us of host time; that step as a whole 25.4 -> 15.6 us)."""
    words = []
    add = words.append
    try:
        for obj in objects:
            nbytes = getattr(obj, "nbytes", None)
            if nbytes.__class__ is int:   # a tensor
                add(obj.data_ptr())
                add(nbytes)
            else:
                buffer = view(obj)
                add(buffer.ptr or 0)
                add(buffer.len_bytes)
    except AttributeError:
        view(obj)   # says what cannot be borrowed
        raise
    if 8 * len(words) != sizeof(struct_type):   # `from_buffer` takes an array that is too long, and later fields would shift
        raise TypeError(f"{struct_type.__name__} takes {len(struct_type._fields_)} buffers, not {len(objects)}")
    return struct_type.from_buffer(array("Q", words))


def stream_handle(stream) -> int:
    """hipStream_t of a torch stream (or the current one); 0 is the legacy default stream."""
    if stream is None:
        import torch

        try:
            # the handle itself; current_stream() builds a Python object around it first
            return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device())
        except AttributeError:   # no public name of torch
            return int(torch.cuda.current_stream().cuda_stream)
    if hasattr(stream, "cuda_stream"):
        return int(stream.cuda_stream)
    return int(stream)


def param_block(block) -> int:
    if block is None:
        return 0
    if hasattr(block, "data_ptr"):
        return int(block.data_ptr())
    return int(block)
