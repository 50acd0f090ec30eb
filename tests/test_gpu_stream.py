"""The launch stream of the host mirror is torch's current stream."""
import pytest
import torch

from sager_amd import ops

pytestmark = pytest.mark.gpu


def test_launch_stream_follows_the_current_stream():
    assert ops._stream() == torch.cuda.current_stream().cuda_stream
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert ops._stream() == side.cuda_stream != 0
    g = torch.cuda.CUDAGraph()
    x = torch.zeros(256, device="cuda")
    q = ops.q8k_empty(1, 256)
    ops.quantize_q8_k(x, out=q)
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        assert ops._stream() == torch.cuda.current_stream().cuda_stream
        ops.quantize_q8_k(x, out=q)
    x.fill_(1.0)
    g.replay()
    want = ops.quantize_q8_k(x)
    torch.cuda.synchronize()
    assert torch.equal(q, want)
