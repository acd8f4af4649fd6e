"""The stream that every launch goes to."""
import pytest
import torch

from dynamo_exp_amd import ops


@pytest.mark.gpu
def test_launches_go_to_the_current_stream():
    """The raw handle is the current stream's: by default, inside other streams, nested, behind them, and under capture."""
    def same():
        return ops._stream() == torch.cuda.current_stream().cuda_stream

    x = torch.zeros(4, device="cuda")
    assert same()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(a):
        assert same() and ops._stream() == a.cuda_stream
        with torch.cuda.stream(b):
            assert same() and ops._stream() == b.cuda_stream
        assert same()
    assert same()
    g = torch.cuda.CUDAGraph()
    with torch.inference_mode(), torch.cuda.graph(g):  # (the generator's state is an inference tensor once an engine has captured)
        assert same()
        x.add_(1)
