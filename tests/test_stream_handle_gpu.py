"""The current-stream handle every operator launches on, against torch's own."""
import threading

import pytest
import torch

from magicube_amd.spmm import _stream, current_stream_handle

pytestmark = pytest.mark.gpu


def test_handle_follows_the_current_stream():
    side = torch.cuda.Stream()
    assert current_stream_handle() == torch.cuda.current_stream().cuda_stream
    with torch.cuda.stream(side):
        assert current_stream_handle() == _stream(None) == side.cuda_stream == _stream(side)
        seen = []
        # a thread has a current stream of its own
        t = threading.Thread(target=lambda: seen.append((current_stream_handle(),
                                                         torch.cuda.current_stream().cuda_stream)))
        t.start()
        t.join()
        assert seen[0][0] == seen[0][1] != side.cuda_stream
    assert current_stream_handle() == torch.cuda.current_stream().cuda_stream
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        x = torch.zeros(4, device="cuda")
        assert current_stream_handle() == side.cuda_stream
        x.add_(1)
    graph.replay()
    torch.cuda.synchronize()
    assert x.tolist() == [1.0] * 4
