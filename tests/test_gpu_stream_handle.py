"""The stream a call without one runs on: the thread's current stream, also
inside a stream context and in a thread of its own."""
import threading

import pytest


@pytest.mark.gpu
def test_current_stream_handle():
    import torch

    from compact_schemes_amd import _stream
    want = lambda: torch.cuda.current_stream().cuda_stream or None
    torch.cuda.init()
    assert _stream().value == want()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert _stream().value == side.cuda_stream == want()
        seen = []
        t = threading.Thread(target=lambda: seen.append((_stream().value, want())))
        t.start()
        t.join()
        assert seen[0][0] == seen[0][1]
    assert _stream().value == want()
    assert _stream(side).value == side.cuda_stream
