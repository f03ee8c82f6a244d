"""The stream that the Python entry points launch on is torch's current one."""
import threading

import pytest

from onenew_amd import hip

pytestmark = pytest.mark.gpu


def test_current_stream():
    import torch
    hip.init(0)
    mine = lambda: hip._stream() == torch.cuda.current_stream().cuda_stream  # noqa: E731
    assert mine()
    seen, streams = [], [torch.cuda.Stream() for _ in range(2)]
    for s in streams:
        with torch.cuda.stream(s):
            assert mine() and hip._stream() == s.cuda_stream
            thread = threading.Thread(target=lambda: seen.append(mine() and hip._stream() != s.cuda_stream))   # a thread starts on the default stream
            thread.start()
            thread.join()
            with torch.cuda.stream(None):
                assert hip._stream() == s.cuda_stream
        assert mine()
    assert seen == [True, True]
    graph, x, y = torch.cuda.CUDAGraph(), torch.arange(64.0, device="cuda"), torch.zeros(64, device="cuda")
    with torch.cuda.graph(graph):
        assert mine()
        hip.copy_f32(x, y)
    for i in range(3):
        x.fill_(float(i))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(x, y)
