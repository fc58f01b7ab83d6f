"""`pack` lays out what one `view` per field would, for everything a buffer can be given as."""
import pytest
import torch

from khalamari_amd._buffers import NO_BUFFER, pack, stream_handle, view
from khalamari_amd._lib import Buffer, RmsNormRopeBuffers, SlicedKvMapBuffers


class Borrowed:
    def data_ptr(self):
        return 4096

    def numel(self):
        return 6

    def element_size(self):
        return 2


def test_packed_fields_equal_the_views():
    tensor = torch.zeros(3, 5, dtype=torch.bfloat16)
    objects = (tensor, tensor[1:], torch.zeros(0, dtype=torch.int32), (1 << 47, 1 << 40), Buffer(64, 16), NO_BUFFER, Borrowed(), torch.nn.Parameter(torch.ones(7)))
    packed = pack(SlicedKvMapBuffers, *objects)
    for (name, _), obj in zip(SlicedKvMapBuffers._fields_, objects):
        expected, actual = view(obj), getattr(packed, name)
        assert (actual.ptr, actual.len_bytes) == (expected.ptr, expected.len_bytes), name


def test_what_is_no_buffer_is_refused():
    with pytest.raises(TypeError, match="cannot borrow"):
        pack(RmsNormRopeBuffers, (1, 2), 7, (1, 2), (1, 2))
    with pytest.raises(TypeError, match="cannot borrow"):
        pack(RmsNormRopeBuffers, (1, 2), None, (1, 2), (1, 2))
    with pytest.raises(TypeError, match="cannot borrow"):
        pack(RmsNormRopeBuffers, (1, 2), memoryview(b"host"), (1, 2), (1, 2))   # counts its bytes, but has no device pointer
    with pytest.raises((TypeError, ValueError)):
        pack(RmsNormRopeBuffers, (1, 2), (1, 2))   # a field is missing


def test_a_surplus_buffer_is_refused():
    # one more object would shift every field behind it: the kernel would get pointers of other buffers
    with pytest.raises(TypeError, match="takes 4 buffers, not 5"):
        pack(RmsNormRopeBuffers, (1, 2), (1, 2), (1, 2), (1, 2), (1, 2))


class CountsItsBytes(Borrowed):
    def nbytes(self):
        return self.numel() * self.element_size()


class BorrowedPair(tuple):
    def data_ptr(self):
        raise AssertionError("a (pointer, bytes) pair is taken as it is")


def test_objects_that_only_view_understands():
    packed = pack(RmsNormRopeBuffers, CountsItsBytes(), BorrowedPair((64, 16)), (-1, 16), (1, 2))
    for (name, _), expected in zip(RmsNormRopeBuffers._fields_, (view(CountsItsBytes()), view(BorrowedPair((64, 16))), view((-1, 16)), view((1, 2)))):
        actual = getattr(packed, name)
        assert (actual.ptr, actual.len_bytes) == (expected.ptr, expected.len_bytes), name


class Stream:
    cuda_stream = 77


def test_current_stream_without_the_raw_handle(monkeypatch):
    # the raw handle is no public name of torch: without it the stream object is asked
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: Stream())
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    assert stream_handle(None) == 77
    assert stream_handle(Stream()) == 77 and stream_handle(5) == 5
