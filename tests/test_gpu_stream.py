"""Launches go to torch's current stream of the operand's device, whichever
stream is current at the call."""

from __future__ import annotations

import pytest
import torch

from sparsecore_amd import _lib

pytestmark = pytest.mark.gpu


def test_stream_of_follows_the_current_stream(dev):
    t = torch.zeros(1, device=dev)
    for stream in (torch.cuda.default_stream(), torch.cuda.Stream(), torch.cuda.Stream()):
        with torch.cuda.stream(stream):
            assert _lib.stream_of(t) == stream.cuda_stream
    assert _lib.stream_of(t) == torch.cuda.current_stream(dev).cuda_stream
