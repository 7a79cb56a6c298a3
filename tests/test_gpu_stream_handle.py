"""stream_handle() is the stream torch would launch on: the default one, a side
stream inside its context and its restoration, per thread."""
from __future__ import annotations

import threading

import pytest
import torch

from pourover_amd import _lib as L

pytestmark = pytest.mark.gpu


def _current():
    h = L.stream_handle().value or 0
    assert h == torch.cuda.current_stream().cuda_stream
    return h


def test_follows_torch():
    torch.zeros(1, device="cuda")
    side = torch.cuda.Stream()
    default = _current()
    with torch.cuda.stream(side):
        assert _current() == side.cuda_stream
        seen = []
        t = threading.Thread(target=lambda: seen.append(_current()))
        t.start()
        t.join()
        assert seen == [default]  # the current stream is a thread's own
    assert _current() == default
    assert L.stream_handle(side).value == side.cuda_stream
