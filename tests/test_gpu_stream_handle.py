"""The stream that calls without one take is torch's current stream."""
import threading

import pytest

from yolohtli_amd.solver import _stream_handle


def _current():
    import torch
    return torch.cuda.current_stream().cuda_stream


@pytest.mark.gpu
def test_default_stream_is_torchs_current_one(torch_cuda):
    import torch
    torch.zeros(1, device="cuda")
    side = torch.cuda.Stream()
    assert _stream_handle(None) == _current()
    assert _stream_handle(side) == side.cuda_stream
    with torch.cuda.stream(side):
        assert _stream_handle(None) == side.cuda_stream == _current()
        seen = []  # another thread's current stream is its own
        t = threading.Thread(target=lambda: seen.append((_stream_handle(None), _current())))
        t.start()
        t.join()
        assert seen[0][0] == seen[0][1] != side.cuda_stream
    assert _stream_handle(None) == _current()


def test_no_stream_without_a_device():
    import torch
    if torch.cuda.is_available():
        pytest.skip("a device is there")
    assert _stream_handle(None) is None
    assert _stream_handle(7) == 7
