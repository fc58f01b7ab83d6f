"""Plans uploaded one after the other while the stream is busy: every step sees its own, on more updates than there are staging blocks."""
import numpy as np
import pytest
import torch

from khalamari_amd import batch_metadata, sdpa, sliced_kv
from khalamari_amd._lib import DTYPE_BF16, KhmError
from khalamari_amd.selector import GQAReplayBucketPolicy, RequestShape, Selector

from . import gpu_runner

pytestmark = pytest.mark.gpu


class _View:
    def __init__(self, buffer):
        self.__cuda_array_interface__ = {"shape": (buffer.len_bytes // 4,), "typestr": "<i4", "data": (buffer.ptr, False), "version": 2}


def _selector(max_tokens):
    return Selector.for_lookup(sdpa.Config(DTYPE_BF16, 32, 8, 128, 16), max_tokens, sliced_kv.Layout(16, 1, 512, 1))


@pytest.mark.parametrize("q_lens", [[1] * 9, [3, 1, 40, 2]])
def test_every_step_sees_its_own_plan(device, q_lens):
    selector = _selector(sum(q_lens))
    limits = selector.limits()
    policy = GQAReplayBucketPolicy(limits.max_tokens, limits.max_map_task_templates)
    metadata = batch_metadata.GQAMetadataBuffers(limits.max_tokens, limits.max_map_task_templates)
    views = [torch.as_tensor(_View(metadata.buffer(i)), device=device) for i in range(6)]
    cu = np.concatenate([[0], np.cumsum(q_lens)]).tolist()
    stream, busy, seen, planned = torch.cuda.Stream(), torch.randn(2048, 2048, device=device), [], []
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        for step in range(8):
            for _ in range(10):
                busy = busy @ busy.clamp(-0.01, 0.01)
            histories = [37 * r + 101 * step for r in range(len(q_lens))]
            selection = selector.select(RequestShape.from_batch(histories, cu), policy, cu[-1])
            metadata.update(list(range(len(q_lens))), histories, cu, selection)
            seen.append([view.clone() for view in views])
            planned.append([metadata.host(i) for i in range(6)])
    stream.synchronize()
    for step, (device_arrays, host_arrays) in enumerate(zip(seen, planned)):
        for i in range(6):
            assert np.array_equal(device_arrays[i].cpu().numpy().view(np.uint32), host_arrays[i]), (step, i)


def test_an_update_is_not_captured(device):
    selector = _selector(4)
    limits = selector.limits()
    metadata = batch_metadata.GQAMetadataBuffers(limits.max_tokens, limits.max_map_task_templates)
    selection = selector.select(RequestShape.from_batch([5, 6, 7, 8], [0, 1, 2, 3, 4]), GQAReplayBucketPolicy(limits.max_tokens, limits.max_map_task_templates), 4)
    refused = []

    def record():
        try:
            metadata.update([0, 1, 2, 3], [5, 6, 7, 8], [0, 1, 2, 3, 4], selection)
        except KhmError as error:
            refused.append(str(error))
        torch.zeros(1, device=device)

    gpu_runner.capture_graph(record)
    assert len(refused) == 1 and "stream wait failed" in refused[0]
    metadata.update([0, 1, 2, 3], [5, 6, 7, 8], [0, 1, 2, 3, 4], selection)
    torch.cuda.synchronize()


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="two GPUs")
@pytest.mark.parametrize("own_stream", [False, True])
def test_an_update_on_a_stream_of_another_device(device, own_stream):
    """The arrays are the first device's; the update is called with the second one current."""
    selector = _selector(4)
    limits = selector.limits()
    with torch.cuda.device(0):
        metadata = batch_metadata.GQAMetadataBuffers(limits.max_tokens, limits.max_map_task_templates)
        views = [torch.as_tensor(_View(metadata.buffer(i)), device="cuda:0") for i in range(6)]
    policy = GQAReplayBucketPolicy(limits.max_tokens, limits.max_map_task_templates)
    with torch.cuda.device(1):
        for step in range(5):
            histories = [step, step + 1, step + 2, step + 3]
            selection = selector.select(RequestShape.from_batch(histories, [0, 1, 2, 3, 4]), policy, 4)
            metadata.update([0, 1, 2, 3], histories, [0, 1, 2, 3, 4], selection, stream=torch.cuda.Stream() if own_stream else None)
            torch.cuda.synchronize()
            for i in range(6):
                assert np.array_equal(views[i].cpu().numpy().view(np.uint32), metadata.host(i)), (step, i)
