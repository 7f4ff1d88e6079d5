"""Calls without a stream argument run on the calling thread's current torch
stream: the default one, inside torch.cuda.stream(), and per thread."""
import threading

import pytest

pytestmark = pytest.mark.gpu


def test_current_stream_handle():
    import torch

    assert torch.cuda.is_available()
    import w4a16_hip as hip

    torch.cuda.init()
    want = torch.cuda.current_stream().cuda_stream
    assert hip._stream(None) == want
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        assert hip._stream(None) == s.cuda_stream
        other = []
        t = threading.Thread(target=lambda: other.append(hip._stream(None)))
        t.start()
        t.join()
        assert other == [want]   # another thread keeps its own current stream
    assert hip._stream(None) == want
    assert hip._stream(s) == s.cuda_stream
