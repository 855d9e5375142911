"""The stream handle of every form of device that torch's own function takes."""

import pytest
import torch

from akv_amd import ops


@pytest.mark.parametrize("device", [torch.device("cuda", 0), torch.device("cuda"), "cuda:0", "cuda", 0, None])
@pytest.mark.parametrize("raw", [True, False])
def test_forms_of_device(monkeypatch, device, raw):
    """On the CPU: torch's functions stood in for, with and without the
    private one (a torch that has none)."""
    asked = []

    class Stream:
        cuda_stream = 1234

    monkeypatch.setattr(torch.cuda, "current_stream", lambda d=None: asked.append(d) or Stream())
    monkeypatch.setattr(ops, "_raw_stream", (lambda index: 1234) if raw else None)
    assert ops.current_stream_handle(device) == 1234
    assert asked == ([] if raw and isinstance(device, torch.device) and device.index is not None else [device])


@pytest.mark.gpu
@pytest.mark.parametrize("form", [torch.device("cuda", 0), torch.device("cuda"), "cuda:0", "cuda", 0, None])
def test_handle_is_the_current_streams(device, form):
    assert ops.current_stream_handle(form) == torch.cuda.current_stream(form).cuda_stream
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        assert ops.current_stream_handle(form) == stream.cuda_stream
