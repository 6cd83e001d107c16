"""The stream handle and the device switch that every call's host side takes."""
import contextlib
import threading

import pytest

pytestmark = pytest.mark.gpu


def test_stream_handle_is_the_current_streams(hrf):
    import torch
    from complex_valued_holographic_radiance_fields_amd import _lib

    dev = torch.zeros(1, device="cuda").device
    side = torch.cuda.Stream()
    assert _lib.stream_ptr(dev) == torch.cuda.current_stream(dev).cuda_stream
    assert _lib.stream_ptr(torch.device("cuda")) == torch.cuda.current_stream().cuda_stream
    with torch.cuda.stream(side):
        assert _lib.stream_ptr(dev) == side.cuda_stream
        seen = []
        th = threading.Thread(target=lambda: seen.append(
            (_lib.stream_ptr(dev), torch.cuda.current_stream(dev).cuda_stream)))
        th.start()
        th.join()
        assert seen[0][0] == seen[0][1]  # another thread has its own current stream
    assert _lib.stream_ptr(dev) != side.cuda_stream


def test_device_switch_only_where_needed(hrf, monkeypatch):
    import torch
    from complex_valued_holographic_radiance_fields_amd import _lib

    dev = torch.device("cuda", torch.cuda.current_device())
    assert isinstance(_lib.on_device(dev), contextlib.nullcontext)
    with _lib.on_device(dev), _lib.on_device(dev):
        assert torch.cuda.current_device() == dev.index
    # any other device (or one without an index) takes torch's own switch
    monkeypatch.setattr(torch.cuda, "current_device", lambda: dev.index + 1)
    assert isinstance(_lib.on_device(dev), torch.cuda.device)
    assert isinstance(_lib.on_device(torch.device("cuda")), torch.cuda.device)
